// RK3's last two stages in one launch, for grids so small that a launch is
// latency: 1D grids above avh_line.hpp's, and small 2D ones.
//
// The second stage needs no number from the rest of the grid but dt, so a
// workgroup can evaluate it on its tile and the halo the third stage wants,
// TX + 2G by TY + 2G cells, from U1 on TX + 4G by TY + 4G, and run the third
// stage on the tile.  The halo's fluxes are evaluated by every workgroup that
// needs them; where a stage launch is mostly latency that costs less than a
// launch.  A thread holds one cell of the U1 region (or a few), U0, U1 and U2
// in registers; the two regions go through LDS.
// U1 is formed from L0 and the copy of U0 that the first stage leaves
// (StageParams::copy), since the launch overwrites the state.  Outside the
// domain U2 is what its boundary image is: with periodic boundaries the same
// operations on the same values give it, with neumann ones it is copied from
// the cell it mirrors, which the region holds.  The boundary map has to take
// cells 2G outside the grid, so no axis is shorter than that (pair_shape).
// Bound by the chain of two flux evaluations and a launch's latency.  us of an
// RK3 step with three stage launches and with two: 2D, weno2, hll3, 16x7 tiles,
// 64^2 15.3 -> 13.9, 128^2 18.2 -> 16.5, 256^2 (where 16x15 on 512 threads
// takes 26.0) 30.5 -> 30.0; tiles of 8x4 13.8 at 64^2 but 15.5 against 14.7 at
// 100x70, of 16x15 17.8 and 32 at 64^2 and 256^2.  1D, tiles of 240 cells,
// against 64 and 256: burgers 12 -> 9.0 (3000 cells), 13.9 -> 9.1 (8192),
// 116 -> 105 (10^6); euler1 18.5 -> 12.8, 20 -> 12.9, 136 -> 112.
#pragma once
#include "avh_stage.hpp"

#pragma clang fp contract(off)

namespace avh {

template <class EQ, int RECON, class FLUX, int DIM, int TX, int TY, int NT>
struct PairKernel {
    typedef typename OpsFor<FLUX::FAST>::type Ops;
    static constexpr int NV = EQ::NV;
    static constexpr int G = ReconTraits<RECON>::GHOST;
    static constexpr int GY = DIM == 2 ? G : 0;
    static constexpr int NTHREADS = NT;

    // a region of cells in LDS: the tile and H rings of G cells around it, and
    // the fluxes of the interfaces of the ring inside it
    template <int H>
    struct Region {
        static constexpr int LX = TX + 2 * G * H, LY = TY + 2 * GY * H, CELLS = LX * LY;
        static constexpr int IX = LX - 2 * G, IY = LY - 2 * GY;  // cells whose fluxes it serves
        static constexpr int NIX = (IX + 1) * IY, NIY = DIM == 2 ? IX * (IY + 1) : 0;
        static constexpr int YT = (NIY + 63) / 64 * 64;  // y items, in whole wavefronts
        static constexpr int NF = NIX + NIY;
    };
    typedef Region<2> R1;  // U1
    typedef Region<1> R2;  // U2
    static constexpr int CPT = (R1::CELLS + NT - 1) / NT;  // cells per thread

    __host__ __device__ static unsigned int tiles(const int* n) {
        return (unsigned int)(((n[0] + TX - 1) / TX) * ((n[1] + TY - 1) / TY));
    }
    template <class OPS, int DIR>
    __device__ __forceinline__ static double interface(const double* u, int vs, int ia, int sd, double gamma, double* F,
                                                       bool& ok) {
        double qa[NV], qb[NV];
        recon_face_ops<RECON, NV, true, OPS>(u, vs, ia, sd, qa);        // right face of a
        recon_face_ops<RECON, NV, false, OPS>(u, vs, ia + sd, sd, qb);  // left face of b
        const typename EQ::All aL = EQ::template make_all_ops<OPS>(qa, gamma, ok);
        const typename EQ::All aR = EQ::template make_all_ops<OPS>(qb, gamma, ok);
        return FLUX::template flux_ops<OPS, DIR, EQ>(aL, aR, gamma, F, ok);
    }
    template <class R, int DIR>
    __device__ __forceinline__ static void flux(const double* u, double* f, int it, double gamma, bool adm) {
        // cell left of the interface, in the region's coordinates
        const int cx = (DIR == 0 ? it % (R::IX + 1) - 1 : it % R::IX) + G;
        const int cy = (DIR == 0 ? it / (R::IX + 1) : it / R::IX - 1) + GY;
        const int ia = cy * R::LX + cx;
        constexpr int SD = DIR == 0 ? 1 : R::LX;
        double F[NV];
        bool ok = adm;
        interface<Ops, DIR>(u, R::CELLS, ia, SD, gamma, F, ok);
        if (FLUX::FAST && !ok) {
            ok = true;
            interface<PlainOps, DIR>(u, R::CELLS, ia, SD, gamma, F, ok);
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) f[v * R::NF + (DIR == 0 ? 0 : R::NIX) + it] = F[v];
    }
    template <class R>
    __device__ __forceinline__ static void fluxes(const double* u, double* f, double gamma, bool adm) {
        for (int it = threadIdx.x; it < R::YT + R::NIX; it += NT) {
            if (DIM == 2 && it < R::YT) {
                if (it < R::NIY) flux<R, DIM == 2 ? 1 : 0>(u, f, it, gamma, adm);
            } else {
                flux<R, 0>(u, f, it - R::YT, gamma, adm);
            }
        }
    }
    // net flux of the cell at (cx, cy) of the cells R serves: 0 + x + y
    template <class R>
    __device__ __forceinline__ static void net(const double* f, int cx, int cy, double* l) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double* const g = f + v * R::NF;
            const int ix = cy * (R::IX + 1) + cx;
            l[v] = 0.0 + ((-g[ix + 1]) + g[ix]);
            if (DIM == 2) {
                const int iy = R::NIX + cy * R::IX + cx;
                l[v] = l[v] + ((-g[iy + R::IX]) + g[iy]);
            }
        }
    }

    // one vote per wavefront through LDS; the barrier publishes the region too
    __device__ __forceinline__ static bool vote(bool adm, int* s_adm) {
        if constexpr (FLUX::FAST) {
            const bool all = __all(adm);
            if ((threadIdx.x & 63) == 0) s_adm[threadIdx.x >> 6] = all;
        }
        lds_barrier();
        if constexpr (FLUX::FAST) {
            int all = s_adm[0];
#pragma unroll
            for (int i = 1; i < NT / 64; ++i) all = all & s_adm[i];
            adm = all != 0;
        }
        return adm;
    }

    // P.in: L0, P.u0: the copy of U0, P.out: the state
    __device__ static void run(const StageParams& P) {
        __shared__ double u1s[NV * R1::CELLS];
        __shared__ double u2s[NV * R2::CELLS];
        __shared__ double f[NV * (R1::NF > R2::NF ? R1::NF : R2::NF)];
        __shared__ int s_adm[2][NT / 64];
        __shared__ double s_ws[3][NT / 64];
        __shared__ StepEnd s_end;
        Control* const ctrl = P.ctrl;
        const int n0 = P.n[0], n1 = P.n[1];
        const long long nc = P.ncells;
        const unsigned int tile = tile_id_xcd(blockIdx.x, gridDim.x);
        const int ntx = (n0 + TX - 1) / TX;
        const int ox = (int)(tile % ntx) * TX, oy = (int)(tile / ntx) * TY;

        double u0[CPT][NV], u1[CPT][NV], u2[CPT][NV];
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = (int)threadIdx.x + m * NT < R1::CELLS ? threadIdx.x + m * NT : R1::CELLS - 1;
            int gx = ox + c % R1::LX - 2 * G, gy = oy + c / R1::LX - 2 * GY;
            gx = bc_map(gx < n0 + 2 * G ? gx : n0 + 2 * G - 1, n0, P.bc);
            gy = DIM == 2 ? bc_map(gy < n1 + 2 * G ? gy : n1 + 2 * G - 1, n1, P.bc) : 0;
            const long long gi = (long long)gy * n0 + gx;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                u1[m][v] = P.in[v * nc + gi];
                u0[m][v] = P.u0[v * nc + gi];
            }
        }
        if (!ctrl->active) return;  // step past the end: no-op
        const double s = stage_scale(P, ctrl, MODE_RK3_3, &s_end);

        // second stage
        const bool g_ok = EQ::gamma_admitted(P.gamma);
        bool adm = g_ok;
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = threadIdx.x + m * NT;
#pragma unroll
            for (int v = 0; v < NV; ++v) u1[m][v] = u1[m][v] * s + u0[m][v];
            if (FLUX::FAST) adm = adm & EQ::admitted(u1[m]);
            if (R1::CELLS % NT != 0 && c >= R1::CELLS) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) u1s[v * R1::CELLS + c] = u1[m][v];
        }
        adm = vote(adm, s_adm[0]);
        fluxes<R1>(u1s, f, P.gamma, adm);
        lds_barrier();
        adm = g_ok;
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = threadIdx.x + m * NT;
            const int cx = c % R1::LX - G, cy = c / R1::LX - GY;  // in R2's coordinates
            const bool here = c < R1::CELLS && cx >= 0 && cx < R2::LX && cy >= 0 && cy < R2::LY;
            double l[NV];
            net<R1>(f, here ? cx : 0, here ? cy : 0, l);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                double o = l[v] * s;
                o = o + u1[m][v];
                o = o * (1. / 3.);
                o = o + u0[m][v];
                o = o * (3. / 4.);
                u2[m][v] = o;
            }
            if (!here) continue;
            // a cell outside the domain: its own value with periodic
            // boundaries, below with neumann ones
            const int gx = ox + cx - G, gy = oy + cy - GY;
            const bool inside = gx >= 0 && gx < n0 && gy >= 0 && gy < n1;
            if (!inside && P.bc != BC_PERIODIC) continue;
            if (FLUX::FAST && gx < n0 + G && gy < n1 + G) adm = adm & EQ::admitted(u2[m]);
#pragma unroll
            for (int v = 0; v < NV; ++v) u2s[v * R2::CELLS + cy * R2::LX + cx] = u2[m][v];
        }
        adm = vote(adm, s_adm[1]);
        if (P.bc != BC_PERIODIC) {
            for (int c = threadIdx.x; c < R2::CELLS; c += NT) {
                const int gx = ox + c % R2::LX - G, gy = oy + c / R2::LX - GY;
                if ((gx >= 0 && gx < n0 && gy >= 0 && gy < n1) || gx >= n0 + G || gy >= n1 + G) continue;
                const int sx = bc_map(gx, n0, P.bc) - ox + G;
                const int sy = DIM == 2 ? bc_map(gy, n1, P.bc) - oy + GY : 0;
#pragma unroll
                for (int v = 0; v < NV; ++v) u2s[v * R2::CELLS + c] = u2s[v * R2::CELLS + sy * R2::LX + sx];
            }
            lds_barrier();
        }

        // third stage; interfaces past the grid's edge work on whatever the
        // region holds there, and no cell takes their fluxes
        fluxes<R2>(u2s, f, P.gamma, adm);
        lds_barrier();
        bool bad = false;
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = threadIdx.x + m * NT;
            const int cx = c % R1::LX - 2 * G, cy = c / R1::LX - 2 * GY;
            if (c >= R1::CELLS || cx < 0 || cx >= TX || cy < 0 || cy >= TY || ox + cx >= n0 || oy + cy >= n1) continue;
            double l[NV], r[NV];
            net<R2>(f, cx, cy, l);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                double o = l[v] * s;
                o = o + u2[m][v];
                o = o * 2.0;
                o = o + u0[m][v];
                o = o * (1. / 3.);
                r[v] = o;
            }
            bad = bad || !EQ::obeys_fast(r, P.gamma);
            const long long gi = (long long)(oy + cy) * n0 + ox + cx;
#pragma unroll
            for (int v = 0; v < NV; ++v) store_through(P.out + v * nc + gi, r[v]);
        }
        end_of_tile<NT>(P, ctrl, MODE_RK3_3, 0.0, 0.0, 0.0, s_ws, bad, s_end);
    }
};

template <class K>
__global__ __launch_bounds__(K::NTHREADS) __attribute__((amdgpu_waves_per_eu(4))) void pair_kernel(StageParams P) {
    K::run(P);
}

}  // namespace avh
