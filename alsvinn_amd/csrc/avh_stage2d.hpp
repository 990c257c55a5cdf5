// Fused FP64 stage kernel for 2D grids: TX x TY tiles staged in LDS.
//
// Steps as listed in avh_stage.hpp: the tile and its halo go to LDS,
// interface fluxes per direction, net flux and RK combination per cell.  What
// is 2D's own is how the work is dealt to threads; the kernel is bound by the
// FP64 pipe on large grids and by the latency of one workgroup's chain on
// small ones.
//   Staging   a thread keeps one column of the tile and takes every NT/LX-th
//             row, so the boundary map of x is evaluated once and that of y
//             once a row.
//   Fluxes    a thread takes STEPS consecutive interfaces of a row (column)
//             and marches along them: of WENO2's smoothness terms each
//             difference is inverted once (4 for 2 interfaces instead of 6),
//             and the item's position is decoded once.  Where both directions
//             fit one turn of the workgroup (DUAL), its wavefronts evaluate
//             them side by side, which halves the chain.
// Measured against one interface at a time with divided tile indices (one
// MI355X, RK3 first plus second stage): 64^2 14.4 -> 9.5 us (16x7 tiles, both
// directions at once; 16x15 tiles 12.6), 2048^2 310 -> 300 us; VALU
// instructions of a 1024^2 stage 18.1 M -> 15.1 M together with SharedOps'
// checks per cell.
#pragma once
#include "avh_stage.hpp"

#pragma clang fp contract(off)

namespace avh {

template <class EQ, int RECON, class FLUX, int TX, int TY, int NT, int MODE_CT = -1>
struct TileKernel2 {
    // the kernels compiled per stage mode index cells with 32-bit values
    // (their launchers take them only for grids of fewer than 2^29 cells)
    static constexpr bool OFF32 = MODE_CT >= 0;
    typedef typename std::conditional<OFF32, unsigned int, long long>::type Idx;
    typedef typename OpsFor<FLUX::FAST>::type Ops;
    static constexpr int NV = EQ::NV;
    static constexpr int G = ReconTraits<RECON>::GHOST;
    static constexpr int LX = TX + 2 * G;
    static constexpr int LY = TY + 2 * G;
    static constexpr int LT = LX * LY;  // tile cells incl. halo
    static constexpr int NIX = (TX + 1) * TY;
    static constexpr int NIY = TX * (TY + 1);
    static constexpr int YT = (NIY + 63) / 64 * 64;  // threads of the y fluxes when DUAL
    static constexpr bool DUAL = YT + NIX <= NT;
    static constexpr int STEPS = NIX <= NT && NIY <= NT ? 1 : 2;
    static constexpr int PX = (TX + STEPS) / STEPS;  // turns of STEPS interfaces along a row
    static constexpr int PY = (TY + STEPS) / STEPS;
    static_assert(PX * TY <= NT && PY * TX <= NT, "one turn per direction");
    static constexpr int NIMAX = NIX > NIY ? NIX : NIY;
    static constexpr int NF = DUAL ? NIX + NIY : NIMAX;  // flux slots in LDS
    static constexpr int TC = TX * TY;
    static constexpr int NTHREADS = NT;
    static constexpr int CPT = (TC + NT - 1) / NT;  // cells per thread
    static constexpr int RPS = NT / LX;             // rows a staging sweep covers
    static constexpr int SW = (LY + RPS - 1) / RPS;

    __host__ __device__ static unsigned int tiles(const int* n) {
        return (unsigned int)(((n[0] + TX - 1) / TX) * ((n[1] + TY - 1) / TY));
    }
    __device__ __forceinline__ static int lidx(int cx, int cy) { return (cy + G) * LX + (cx + G); }

    // WENO2 under SharedOps: 1/d of the difference between cells i and i + sd
    static constexpr bool RECIPS = RECON == RECON_WENO2 && Ops::SHARED;
    __device__ __forceinline__ static double recip(const double* su, int i, int sd) {
        return RECIPS ? weno2_recip(su[i + sd] - su[i]) : 0.0;
    }

    // flux between cells ia and ia + SD; ra, rb, rc as recip() of the
    // differences before, across and behind the interface (RECIPS only)
    template <class OPS, int DIR>
    __device__ __forceinline__ static double interface(const double* su, int ia, double ra, double rb, double rc,
                                                       double gamma, double* F, bool& ok) {
        constexpr int SD = DIR == 0 ? 1 : LX;
        double qa[NV], qb[NV];
        if constexpr (RECON == RECON_WENO2 && OPS::SHARED) {
            weno2_face_recips<NV, true>(su, LT, ia, SD, rb, ra, qa);
            weno2_face_recips<NV, false>(su, LT, ia + SD, SD, rc, rb, qb);
        } else {
            recon_face_ops<RECON, NV, true, OPS>(su, LT, ia, SD, qa);        // right face of a
            recon_face_ops<RECON, NV, false, OPS>(su, LT, ia + SD, SD, qb);  // left face of b
        }
        const typename EQ::All aL = EQ::template make_all_ops<OPS>(qa, gamma, ok);
        const typename EQ::All aR = EQ::template make_all_ops<OPS>(qb, gamma, ok);
        return FLUX::template flux_ops<OPS, DIR, EQ>(aL, aR, gamma, F, ok);
    }

    // Fluxes of turn `it` along DIR into sf.  A FAST flux evaluates each
    // interface with SharedOps; those whose operands fall outside its range
    // are redone with PlainOps in a second loop, after the first one's
    // registers are free.  `adm`: every cell of the tile is admitted.
    template <int DIR>
    __device__ __forceinline__ static void flux_turn(const double* su, double* sf, int it, int ox, int oy,
                                                     const int* n, double gamma, bool adm, double& ws) {
        constexpr int SD = DIR == 0 ? 1 : LX;
        constexpr int NK = DIR == 0 ? TX + 1 : TY + 1;  // interfaces of a row (column)
        const int k0 = (DIR == 0 ? it % PX : it / TX) * STEPS;
        const int cx = DIR == 0 ? k0 - 1 : it % TX;
        const int cy = DIR == 0 ? it / PX : k0 - 1;
        if (it >= (DIR == 0 ? PX * TY : PY * TX)) return;
        if ((DIR == 0 ? oy + cy : ox + cx) >= n[1 - DIR]) return;
        // interfaces of this turn inside the tile and the grid
        const int here = DIR == 0 ? n[0] - (ox + cx) : n[1] - (oy + cy);
        const int left = NK - k0 < here ? NK - k0 : here;
        const int steps = left < STEPS ? left : STEPS;
        const int slot = DIR == 0 ? cy * (TX + 1) + k0 : k0 * TX + cx;
        constexpr int DS = DIR == 0 ? 1 : TX;
        const int i0 = lidx(cx, cy);
        unsigned int redo = 0;
        double ra = 0.0, rb = 0.0;
        if (steps > 0) {
            ra = recip(su, i0 - SD, SD);
            rb = recip(su, i0, SD);
        }
#pragma unroll 1
        for (int m = 0; m < steps; ++m) {
            const int ia = i0 + m * SD;
            const double rc = recip(su, ia + SD, SD);
            double F[NV];
            bool ok = adm;
            const double w = interface<Ops, DIR>(su, ia, ra, rb, rc, gamma, F, ok);
            if (ok) ws = ws_max(ws, w);
            else redo |= 1u << m;
#pragma unroll
            for (int v = 0; v < NV; ++v) sf[v * NF + slot + m * DS] = F[v];
            ra = rb;
            rb = rc;
        }
        if (FLUX::FAST && redo != 0) {
            for (int m = 0; m < steps; ++m) {
                if (!((redo >> m) & 1u)) continue;
                double F[NV];
                bool ok = true;
                ws = ws_max(ws, interface<PlainOps, DIR>(su, i0 + m * SD, 0.0, 0.0, 0.0, gamma, F, ok));
#pragma unroll
                for (int v = 0; v < NV; ++v) sf[v * NF + slot + m * DS] = F[v];
            }
        }
    }

    template <int DIR>
    __device__ __forceinline__ static void accumulate(const double* sf, double (&acc)[CPT][NV]) {
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = threadIdx.x + m * NT;
            if (TC % NT != 0 && c >= TC) continue;
            const int cx = c % TX, cy = c / TX;
            const int ip = DIR == 0 ? cy * (TX + 1) + cx + 1 : (cy + 1) * TX + cx;
            constexpr int STEP = DIR == 0 ? 1 : TX;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double fp = sf[v * NF + ip];
                const double fm = sf[v * NF + ip - STEP];
                // temp = -F; out[i] += temp[i] + (-1)*temp[i-1]
                acc[m][v] = acc[m][v] + ((-fp) + fm);
            }
        }
    }

    __device__ static void run(const StageParams& P) { run_tile<false, true>(P, tile_id_xcd(blockIdx.x, gridDim.x)); }
    __device__ static void run_volume(const StageParams& P, const VolumeParams& V) {
        run_tile<true>(P, tile_id_xcd(blockIdx.x, gridDim.x), &V);
    }

    // VOL: the cells live in a reference Volume (V; MODE_FLUX_ONLY, or
    // MODE_RK3_3 for the combination V describes) and P.n is the extent of the
    // box the launch covers; otherwise in the interior-only buffers of P
    // with the boundary map for the halo.  LOAD_FIRST: on
    // grids that are not large the test whether the step runs at all comes after
    // the tile's addresses (a single grid's steps nearly always do; of a batch's
    // samples many may have ended).
    template <bool VOL = false, bool LOAD_FIRST = false>
    __device__ static void run_tile(const StageParams& P, const unsigned int tile, const VolumeParams* V = nullptr) {
        __shared__ double su[NV * LT];
        __shared__ double sf[NV * NF];
        __shared__ double s_ws[3][NT / 64];
        __shared__ StepEnd s_end;
        __shared__ int s_adm[NT / 64];

        Control* ctrl = P.ctrl;
        const int mode = MODE_CT >= 0 ? MODE_CT : P.mode;
        // A step past the end is a no-op.  A run is launched in chunks, and most
        // of its last one may lie past the end; on large grids the test comes first:
        // 48 steps past the end of 2048^2 take 980 us with the addresses ahead of
        // it and 495 so, a step before it 871 either way.  Up to some rounds of
        // tiles the addresses ahead are worth more than they cost: at 1024^2 (2310
        // tiles) 397 us against 264, but a step 130.1 us against 131.6 on one
        // card, 122.4 both on another; at 1448^2 (4462) 595 and 340, steps alike.
        // (The shapes that evaluate both directions at once are for small grids.)
        if (!VOL && !(LOAD_FIRST && (DUAL || gridDim.x <= 4096)) && !ctrl->active && mode != MODE_FLUX_ONLY) return;
        const int n0 = P.n[0], n1 = P.n[1];
        const int ntx = (n0 + TX - 1) / TX;
        const int ox = (int)(tile % ntx) * TX, oy = (int)(tile / ntx) * TY;
        const long long nc = P.ncells;
        const bool otf = on_the_fly(mode);

        // 1. stage input tile + halo into LDS through the boundary map.  All
        // loads are issued before the first is used; rows past the tile
        // repeat the last one and are not written.
        const int lx = threadIdx.x % LX, ly0 = threadIdx.x / LX;
        const bool stages = ly0 < RPS;
        int gx = ox + lx - G;
        gx = gx < n0 + G ? gx : n0 + G - 1;
        if (!VOL) gx = bc_map(gx, n0, P.bc);
        Idx sg[SW];
#pragma unroll
        for (int k = 0; k < SW; ++k) {
            const int ly = ly0 + k * RPS < LY ? ly0 + k * RPS : LY - 1;
            int gy = oy + ly - G;
            gy = gy < n1 + G ? gy : n1 + G - 1;
            if constexpr (VOL) sg[k] = volume_index(*V, gx, gy, 0);
            else sg[k] = (Idx)bc_map(gy, n1, P.bc) * n0 + gx;
        }
        double sv[SW][NV], s0[SW][NV];
#pragma unroll
        for (int k = 0; k < SW; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                if constexpr (VOL) sv[k][v] = V->in[v][sg[k]];
                else sv[k][v] = soa_ld<OFF32>(P.in, nc, v, sg[k]);
            }
        if (otf) {
#pragma unroll
            for (int k = 0; k < SW; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) s0[k][v] = soa_ld<OFF32>(P.u0, nc, v, sg[k]);
        }
        if (!VOL && LOAD_FIRST && !ctrl->active && mode != MODE_FLUX_ONLY) return;
        // dt / dx, formed while the loads are in flight
        const double s = (mode == MODE_FLUX_ONLY || mode == MODE_L) ? 0.0
                         : VOL                                       ? V->s
                                                                     : stage_scale(P, ctrl, mode, &s_end);
        if (otf) {
#pragma unroll
            for (int k = 0; k < SW; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) sv[k][v] = sv[k][v] * s + s0[k][v];
        }
#pragma unroll
        for (int k = 0; k < SW; ++k) {
            const int ly = ly0 + k * RPS;
            if (!stages || ly >= LY) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) su[v * LT + ly * LX + lx] = sv[k][v];
        }
        // whether SharedOps may run on this tile: one vote per wavefront
        // through LDS, read by all after the barrier that publishes the tile
        bool adm = EQ::gamma_admitted(P.gamma);
        if constexpr (FLUX::FAST) {
#pragma unroll
            for (int k = 0; k < SW; ++k) adm = adm & EQ::admitted(sv[k]);
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

        double acc[CPT][NV];
#pragma unroll
        for (int m = 0; m < CPT; ++m)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[m][v] = 0.0;
        double ws[2] = {0.0, 0.0};

        // 2./3. interface fluxes into LDS, then x and y accumulated
        if constexpr (DUAL) {
            if (threadIdx.x < YT) flux_turn<1>(su, sf + NIX, threadIdx.x, ox, oy, P.n, P.gamma, adm, ws[1]);
            else flux_turn<0>(su, sf, threadIdx.x - YT, ox, oy, P.n, P.gamma, adm, ws[0]);
            lds_barrier();
            accumulate<0>(sf, acc);
            accumulate<1>(sf + NIX, acc);
        } else {
            flux_turn<0>(su, sf, threadIdx.x, ox, oy, P.n, P.gamma, adm, ws[0]);
            lds_barrier();
            accumulate<0>(sf, acc);
            lds_barrier();
            flux_turn<1>(su, sf, threadIdx.x, ox, oy, P.n, P.gamma, adm, ws[1]);
            lds_barrier();
            accumulate<1>(sf, acc);
        }

        // 4. RK combination and write-back; the U0 loads of all the thread's
        // cells are issued first (cells outside the grid load element 0 and
        // write nothing)
        bool bad = false;
        const bool final_stage = !VOL && (mode == MODE_RK2_2 || mode == MODE_RK3_3);
        const bool combine = !(mode == MODE_FLUX_ONLY || mode == MODE_L);
        Idx gc[CPT];
        bool inside[CPT];
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = threadIdx.x + m * NT;
            const int x = ox + c % TX, y = oy + c / TX;
            inside[m] = (TC % NT == 0 || c < TC) && x < n0 && y < n1;
            if constexpr (VOL) gc[m] = inside[m] ? volume_index(*V, x, y, 0) : 0;
            else gc[m] = inside[m] ? (Idx)y * n0 + x : 0;
        }
        const double ca = VOL ? V->ca : (mode == MODE_RK3_2 ? 1. / 3. : (mode == MODE_RK3_3 ? 2.0 : 1.0));
        const double cb = VOL ? V->cb : (mode == MODE_RK2_2 ? 0.5 : (mode == MODE_RK3_2 ? 3. / 4. : 1. / 3.));
        double u0c[CPT][NV];
        if (combine) {
#pragma unroll
            for (int m = 0; m < CPT; ++m)
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    if constexpr (VOL) u0c[m][v] = V->u0[v][gc[m]];
                    else u0c[m][v] = soa_ld<OFF32>(P.u0, nc, v, gc[m]);
                }
        }
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            if (!inside[m]) continue;
            const int c = threadIdx.x + m * NT;
            const int li = lidx(c % TX, c / TX);
            double r[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double l = acc[m][v];
                if (!combine) {
                    r[v] = l;
                } else {
                    // ((L*s + U) * ca + U0) * cb; the factor 1 of the RK2
                    // stage is exact, so every mode keeps its own rounding
                    double o = l * s;
                    o = o + su[v * LT + li];
                    o = o * ca;
                    o = o + u0c[m][v];
                    o = o * cb;
                    r[v] = o;
                }
            }
            if (final_stage) bad = bad || !EQ::obeys_fast(r, P.gamma);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                if constexpr (VOL) store_through(V->out[v] + gc[m], r[v]);
                else soa_st<OFF32, true>(P.out, nc, v, gc[m], r[v]);
            }
            if (mode == MODE_L && P.copy) {
#pragma unroll
                for (int v = 0; v < NV; ++v) soa_st<OFF32, true>(P.copy, nc, v, gc[m], su[v * LT + li]);
            }
        }
        if (!VOL || mode == MODE_FLUX_ONLY) end_of_tile<NT>(P, ctrl, mode, ws[0], ws[1], 0.0, s_ws, bad, s_end);
    }
};

}  // namespace avh
