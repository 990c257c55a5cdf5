// Fused FP64 stage kernel for 3D grids: a TX x TY column tile marches along z.
//
// Per z-plane k of its chunk [z0, z1) a workgroup
//   * writes plane k (its own columns from registers, the x/y halo ring from
//     HBM through the boundary map) into an LDS plane buffer,
//   * evaluates the x- and y-interface fluxes of the plane from LDS (one work
//     item per interface, as in the 2D kernel) and accumulates them per cell,
//   * evaluates the z-interface flux F(k+1/2) of each column in registers from
//     a sliding window of planes [k+1-HW, k+1+HW] and the right face of
//     plane k kept from the previous iteration; F(k-1/2) is likewise kept,
//   * adds ((-F_z(k+1/2)) + F_z(k-1/2)) after the x and y terms -- the same
//     x, y, z accumulation order as NumericalFluxCPU::computeFlux
//     (alsfvm/src/numflux/NumericalFluxCPU.cpp:170-221) -- and applies the RK
//     stage combination.
// Each plane is read once per workgroup plus its x/y halo ring; no z halo is
// ever reloaded, and the tile has no z-direction quantisation loss.
#pragma once
#include "avh_stage.hpp"

#pragma clang fp contract(off)

namespace avh {

// ENO / WENO2 / none on a register window: u[i][v], stencil centre `c`
// (compile-time), unit stride.  Selects replace ENO's data-dependent index.
// The plain arithmetic; recon_faces_reg has the SharedOps form of WENO2.
template <int RECON, int NV, bool RIGHT, int WZ>
__device__ __forceinline__ void recon_face_reg(const double (&u)[WZ][NV], const int c, double* out) {
    if (RECON == RECON_NONE) {
#pragma unroll
        for (int v = 0; v < NV; ++v) out[v] = u[c][v];
    } else if (RECON == RECON_WENO2) {
        const double eps = 1e-8;
        const double w0 = u[c][0];
        const double dp = u[c + 1][0] - w0;
        const double b0 = dp * dp;
        const double dm = w0 - u[c - 1][0];
        const double b1 = dm * dm;
        const double d0 = 3 * (eps + b0) * (eps + b0);
        const double d1 = 3 * (eps + b1) * (eps + b1);
        if (RIGHT) {
            const double a0 = 2 / d0;
            const double a1 = 1 / d1;
            double w0r, w1r;
            weno2_weights(a0, a1, w0r, w1r);
#pragma unroll
            for (int v = 0; v < NV; ++v)
                out[v] = 0.5 * (w0r * u[c + 1][v] + (3 * w1r + w0r) * u[c][v] - w1r * u[c - 1][v]);
        } else {
            const double a0 = 1 / d0;
            const double a1 = 2 / d1;
            double w0l, w1l;
            weno2_weights(a0, a1, w0l, w1l);
#pragma unroll
            for (int v = 0; v < NV; ++v)
                out[v] = 0.5 * (w1l * u[c - 1][v] + (3 * w0l + w1l) * u[c][v] - w0l * u[c + 1][v]);
        }
    } else {
        constexpr int ORDER = RECON == RECON_ENO2 ? 2 : 3;
        int shift = 0;
        {
            const double ddr = u[c + 1][0] - u[c][0];
            const double ddl = u[c][0] - u[c - 1][0];
            if (fabs(ddl) < fabs(ddr)) shift++;
        }
        if (ORDER == 3) {
            const double d0p = u[c + 2 < WZ ? c + 2 : WZ - 1][0] - u[c + 1][0];
            const double d00 = u[c + 1][0] - u[c][0];
            const double d0m = u[c][0] - u[c - 1][0];
            const double ddr = d0p - d00;
            const double ddl = d00 - d0m;
            if (fabs(ddl) < fabs(ddr)) shift++;
        }
        const int r = RIGHT ? shift + 1 : shift;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < ORDER; ++j) {
                // value at offset j - shift, shift in [0, ORDER-1]
                double val = u[c + j][v];
#pragma unroll
                for (int sft = 1; sft < ORDER; ++sft) {
                    const int idx = c + j - sft;
                    val = (shift == sft) ? u[idx < 0 ? 0 : idx][v] : val;
                }
                acc += eno_coef<ORDER>(r, j) * val;
            }
            out[v] = acc;
        }
    }
}

// Both faces of the window's cell c.  WENO2 under SharedOps: rb comes in as
// 1/d of the difference behind the cell and goes out as 1/d of the one ahead
// (weno2_recip), which is the one behind the next cell of the march, so each
// difference is inverted once.
template <int RECON, int NV, int WZ, class OPS>
__device__ __forceinline__ void recon_faces_reg(const double (&u)[WZ][NV], const int c, double& rb, double* outl,
                                                double* outr) {
    if constexpr (RECON == RECON_WENO2 && OPS::SHARED) {
        const double r1 = rb;
        const double r0 = weno2_recip(u[c + 1][0] - u[c][0]);
        double h0l, h1l, h0r, h1r;
        weno2_half_weights<false>(r0, r1, h0l, h1l);
        weno2_half_weights<true>(r0, r1, h0r, h1r);
        const double hl = 3 * h0l + h1l;
        const double hr = 3 * h1r + h0r;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            outl[v] = h1l * u[c - 1][v] + hl * u[c][v] - h0l * u[c + 1][v];
            outr[v] = h0r * u[c + 1][v] + hr * u[c][v] - h1r * u[c - 1][v];
        }
        rb = r0;
    } else {
        recon_face_reg<RECON, NV, false, WZ>(u, c, outl);
        recon_face_reg<RECON, NV, true, WZ>(u, c, outr);
    }
}

// The plane tile is double-buffered and the x- and y-interface fluxes have LDS
// buffers of their own, so a plane takes two barriers (plane published; fluxes
// published) and its x, y and z flux evaluations run in one barrier-free
// stretch.  A workgroup marches through P.lz planes.
// MODE_CT >= 0 compiles the kernel for that StageMode alone (P.mode must
// equal it): the other modes' branches and registers drop out.
// VOL: the cells live in a reference Volume (V; MODE_FLUX_ONLY, or
// MODE_RK3_3 for the combination V describes) and P.n is the extent of the box
// the launch covers; otherwise in the interior-only buffers of P with the
// boundary map for the halo.
template <class EQ, int RECON, class FLUX, int TX, int TY, int NTH, int MODE_CT = -1, bool VOL = false>
struct MarchKernel3 {
    static constexpr int NV = EQ::NV;
    // Wavefronts a SIMD has to hold.  HLL3's first stage without reconstruction
    // takes 183 registers with R(k) beside the window it equals and 173 without:
    // two wavefronts; held to 168 it spills 5, and three run (first stage at
    // 256^3 757 -> 717 us, 320^3 1465 -> 1385).
    static constexpr int WAVES = RECON == RECON_NONE && MODE_CT == MODE_L ? 3 : 1;
    static constexpr int NC = TX * TY;  // columns: one per thread, threads past them work on the planes only
    static constexpr int NT = NTH;
    static_assert(NT >= NC && NT % 64 == 0, "one thread per column, whole wavefronts");
    static constexpr int G = ReconTraits<RECON>::GHOST;
    static constexpr int HW = G - 1 > 1 ? G - 1 : 1;  // z-window half width
    static constexpr int WZ = 2 * HW + 1;              // planes k+1-HW .. k+1+HW
    static constexpr int LXP = TX + 2 * G;
    static constexpr int LYP = TY + 2 * G;
    static constexpr int LP = LXP * LYP;  // plane cells incl. halo
    static constexpr int NIX = (TX + 1) * TY;
    static constexpr int NIY = TX * (TY + 1);
    static constexpr int NIMAX = NIX > NIY ? NIX : NIY;
    static constexpr int NHALO = LP - TX * TY;

    __host__ __device__ static unsigned int tiles(const int* n, int lz) {
        return (unsigned int)(((n[0] + TX - 1) / TX) * ((n[1] + TY - 1) / TY) * ((n[2] + lz - 1) / lz));
    }

    // Cell indices.  The kernels compiled for the first two RK3 stages index
    // with 32-bit values (their launcher takes them only for grids of fewer
    // than 2^29 cells, so byte offsets stay below 2^32): each load is then a
    // 32-bit offset from a variable's base held in scalar registers, with no
    // 64-bit address arithmetic per lane.  (The final stage, which also
    // stores, runs out of scalar registers that way and is slower.)
    static constexpr bool OFF32 = !VOL && (MODE_CT == MODE_L || MODE_CT == MODE_RK3_2);
    typedef typename std::conditional<OFF32, unsigned int, long long>::type Idx;
    // rows and planes of the buffers, and where cell (0, 0, 0) of the box lies
    struct Layout {
        Idx origin, row, plane;
        __device__ __forceinline__ Idx at(int x, int y, int z) const { return origin + z * plane + y * row + x; }
    };
    __device__ __forceinline__ static Layout layout(const StageParams& P, const VolumeParams* V) {
        if constexpr (VOL) return Layout{volume_index(*V, 0, 0, 0), V->tot[0], (Idx)V->tot[0] * V->tot[1]};
        else return Layout{0, (Idx)P.n[0], (Idx)P.n[0] * P.n[1]};
    }
    __device__ __forceinline__ static double ld_in(const StageParams& P, const VolumeParams* V, int v, Idx gi) {
        if constexpr (VOL) return V->in[v][gi];
        else return soa_ld<OFF32>(P.in, P.ncells, v, gi);
    }
    __device__ __forceinline__ static double ld_u0(const StageParams& P, const VolumeParams* V, int v, Idx gi) {
        if constexpr (VOL) return V->u0[v][gi];
        else return soa_ld<OFF32>(P.u0, P.ncells, v, gi);
    }
    // coordinate g of the buffers for a cell at most G outside the box
    __device__ __forceinline__ static int map_in(int g, int n, int bc) {
        g = g < n + G ? g : n + G - 1;
        return VOL ? g : bc_map(g, n, bc);
    }
    // as map_in along z, where a window wider than the stencil (HW > G - 1)
    // may reach further out; those planes are not used
    __device__ __forceinline__ static int map_z(int g, int n, int bc) {
        if constexpr (VOL) {
            g = g > -G ? g : -G;
            return g < n + G ? g : n + G - 1;
        } else {
            return bc_map(g, n, bc);
        }
    }

    // one input value at a cell; in the on-the-fly stage U0's values are also
    // written to `keep` (stride NC) when given
    __device__ __forceinline__ static void fetch(const StageParams& P, const VolumeParams* V, bool otf, double s,
                                                 Idx gi, double* q, double* keep = nullptr) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double val = ld_in(P, V, v, gi);
            if (otf) {
                const double u = ld_u0(P, V, v, gi);
                if (keep) keep[v * NC] = u;
                val = val * s + u;
            }
            q[v] = val;
        }
    }

    // A kernel compiled for an on-the-fly stage (U1 = L0*s + U0 formed as
    // the tile loads) reads the column's U0 with each window plane; its RK
    // combination needs the same U0 again RING planes later, by which time
    // the line has left L2.  A thread-private LDS ring of RING planes keeps
    // it, where LDS still allows two workgroups per CU (the register budget
    // allows no more).
    static constexpr int RING = 2 + HW;
    static constexpr int LDS_BASE =
        8 * (2 * NV * LP + 2 * NV * NIMAX + 3 * (NT / 64)) + 8 * (NT / 64) + (int)sizeof(StepEnd);
    static constexpr bool U0RING = on_the_fly(MODE_CT) && LDS_BASE + 8 * RING * NV * NC <= 80 * 1024;

    // interface between plane cells ia and ia + SD under OPS
    template <class OPS, int DIR>
    __device__ __forceinline__ static double plane_interface(const double* sp, int ia, int SD, double gamma,
                                                             double* F, bool& ok) {
        double qa[NV], qb[NV];
        recon_face_ops<RECON, NV, true, OPS>(sp, LP, ia, SD, qa);
        recon_face_ops<RECON, NV, false, OPS>(sp, LP, ia + SD, SD, qb);
        const typename EQ::All aL = EQ::template make_all_ops<OPS>(qa, gamma, ok);
        const typename EQ::All aR = EQ::template make_all_ops<OPS>(qb, gamma, ok);
        return FLUX::template flux_ops<OPS, DIR, EQ>(aL, aR, gamma, F, ok);
    }

    template <int DIR>
    __device__ __forceinline__ static bool plane_item(int it, int ox, int oy, const int* n, int& ia) {
        int cx, cy;
        if (DIR == 0) {
            cx = it % (TX + 1) - 1;
            cy = it / (TX + 1);
        } else {
            cx = it % TX;
            cy = it / TX - 1;
        }
        ia = (cy + G) * LXP + (cx + G);
        return (ox + cx < n[0]) && (oy + cy < n[1]);
    }

    // A FAST flux evaluates each interface with SharedOps and redoes those
    // whose operands leave the guarded range with PlainOps (as the 2D stage
    // kernel's flux_turn); otherwise PlainOps throughout.
    // `adm`: every cell of the plane tile is admitted to SharedOps.
    template <int DIR>
    __device__ __forceinline__ static void plane_pass(const double* sp, double* sf, int ox, int oy, const int* n,
                                                      double gamma, bool adm, double& ws) {
        constexpr int NI = DIR == 0 ? NIX : NIY;
        constexpr int SD = DIR == 0 ? 1 : LXP;
        static_assert((NI + NT - 1) / NT <= 32, "one redo bit per turn");
        typedef typename OpsFor<FLUX::FAST>::type Ops;
        unsigned int redo = 0;
        int m = 0;
        for (int it = threadIdx.x; it < NI; it += NT, ++m) {
            int ia;
            if (!plane_item<DIR>(it, ox, oy, n, ia)) continue;
            double F[NV];
            bool ok = adm;
            const double w = plane_interface<Ops, DIR>(sp, ia, SD, gamma, F, ok);
            if (ok) ws = ws_max(ws, w);
            else redo |= 1u << m;
#pragma unroll
            for (int v = 0; v < NV; ++v) sf[v * NIMAX + it] = F[v];
        }
        if (FLUX::FAST && redo != 0) {
            m = 0;
            for (int it = threadIdx.x; it < NI; it += NT, ++m) {
                int ia;
                if (!((redo >> m) & 1u) || !plane_item<DIR>(it, ox, oy, n, ia)) continue;
                double F[NV];
                bool ok = true;
                ws = ws_max(ws, plane_interface<PlainOps, DIR>(sp, ia, SD, gamma, F, ok));
#pragma unroll
                for (int v = 0; v < NV; ++v) sf[v * NIMAX + it] = F[v];
            }
        }
    }

    __device__ static void run(const StageParams& P, const VolumeParams* V = nullptr) {
        __shared__ double sp_buf[2][NV * LP];
        __shared__ double sfx[NV * NIMAX];
        __shared__ double sfy[NV * NIMAX];
        __shared__ double s_ws[3][NT / 64];
        __shared__ StepEnd s_end;
        __shared__ double su0[U0RING ? RING * NV * NC : 1];
        __shared__ int s_adm[2][NT / 64];

        Control* ctrl = P.ctrl;
        const int mode = MODE_CT >= 0 ? MODE_CT : P.mode;
        if (!VOL && !ctrl->active && mode != MODE_FLUX_ONLY) return;

        const int n0 = P.n[0], n1 = P.n[1], n2 = P.n[2];
        const int ntx = (n0 + TX - 1) / TX, nty = (n1 + TY - 1) / TY;
        const unsigned int tile = tile_id_xcd(blockIdx.x, gridDim.x);
        const int tx = tile % ntx;
        const int ty = (tile / ntx) % nty;
        const int tz = tile / (ntx * nty);
        const int ox = tx * TX, oy = ty * TY, z0 = tz * P.lz;
        const int z1 = (z0 + P.lz < n2) ? z0 + P.lz : n2;
        const bool otf = on_the_fly(mode);
        const double s = (mode == MODE_FLUX_ONLY || mode == MODE_L) ? 0.0
                         : VOL                                       ? V->s
                                                                     : stage_scale(P, ctrl, mode, &s_end);
        const Layout lay = layout(P, V);

        // this thread's column.  A column past the grid edge (partial tile)
        // sits where the tile's x/y halo lies, so it loads the boundary image
        // of that position, exactly as the halo ring does.
        const bool has_col = (int)threadIdx.x < NC;
        const int cx = threadIdx.x % TX, cy = has_col ? (int)threadIdx.x / TX : 0;
        const bool col_ok = has_col && (ox + cx < n0) && (oy + cy < n1);
        const int gxc = map_in(ox + cx, n0, P.bc);
        const int gyc = map_in(oy + cy, n1, P.bc);

        double ws[3] = {0.0, 0.0, 0.0};
        double w[WZ][NV];
        double rprev[NV], fprev[NV];
        double rb = 0.0;  // 1/d of the difference behind the next z-reconstructed cell (WENO2)
        // whether SharedOps may run on this column: every cell its window has
        // held is admitted (a column that meets one that is not stays with
        // PlainOps to the end of the chunk)
        bool col_adm = EQ::gamma_admitted(P.gamma);
#pragma unroll
        for (int i = 0; i < WZ; ++i)
#pragma unroll
            for (int v = 0; v < NV; ++v) w[i][v] = 0.0;
#pragma unroll
        for (int v = 0; v < NV; ++v) rprev[v] = fprev[v] = 0.0;

        // prologue: window centred at z0-1 -> R(z0-1); then centred at z0 ->
        // L(z0), R(z0), F_z(z0-1/2); then centred at z0+1 for the loop
        // ring slot of the column's plane p (z0 <= p): U0 at (p - z0) % RING
        const bool ring = U0RING && col_ok;
        double* const su0c = su0 + (U0RING ? threadIdx.x : 0);
        auto slot = [&](int p) { return su0c + ((p - z0) % RING) * NV * NC; };
        if (has_col) {
#pragma unroll
            for (int i = 0; i < WZ; ++i) {
                const int gz = map_z(z0 - 1 - HW + i, n2, P.bc);
                fetch(P, V, otf, s, lay.at(gxc, gyc, gz), w[i], (ring && i > HW) ? slot(z0 - 1 - HW + i) : nullptr);
            }
            double rm1[NV];
            recon_face_reg<RECON, NV, true, WZ>(w, HW, rm1);
#pragma unroll
            for (int i = 0; i < WZ - 1; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) w[i][v] = w[i + 1][v];
            fetch(P, V, otf, s, lay.at(gxc, gyc, map_z(z0 + HW, n2, P.bc)), w[WZ - 1],
                  ring ? slot(z0 + HW) : nullptr);
            if constexpr (FLUX::FAST) {
#pragma unroll
                for (int i = 0; i < WZ; ++i) col_adm = col_adm & EQ::admitted(w[i]);
            }
            if (col_ok) {
                double l0[NV];
                recon_face_reg<RECON, NV, false, WZ>(w, HW, l0);
                recon_face_reg<RECON, NV, true, WZ>(w, HW, rprev);
                const typename EQ::All aL = EQ::make_all(rm1, P.gamma);
                const typename EQ::All aR = EQ::make_all(l0, P.gamma);
                const double wz = FLUX::template flux<2, EQ>(aL, aR, P.gamma, fprev);
                ws[2] = ws_max(ws[2], wz);
            }
#pragma unroll
            for (int i = 0; i < WZ - 1; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) w[i][v] = w[i + 1][v];
            fetch(P, V, otf, s, lay.at(gxc, gyc, map_z(z0 + 1 + HW, n2, P.bc)), w[WZ - 1],
                  ring ? slot(z0 + 1 + HW) : nullptr);
            if (FLUX::FAST && RECON == RECON_WENO2) rb = weno2_recip(w[HW][0] - w[HW - 1][0]);
        }

        bool bad = false;
        const bool final_stage = !VOL && (mode == MODE_RK2_2 || mode == MODE_RK3_3);
        // This thread's cells of the x/y halo ring (HPT per thread at most):
        // their LDS slots and boundary-mapped positions in a plane do not
        // change with k.  The ring rows above and below the tile come first,
        // then the side columns.
        constexpr int HPT = (NHALO + NT - 1) / NT;
        int halo_lds[HPT];
        Idx halo_xy[HPT];
        bool has_halo[HPT];
#pragma unroll
        for (int j = 0; j < HPT; ++j) {
            const int h = threadIdx.x + j * NT;
            has_halo[j] = h < NHALO;
            halo_lds[j] = 0;
            halo_xy[j] = 0;
            if (has_halo[j]) {
                int lx, ly;
                if (h < G * LXP) {
                    ly = h / LXP;
                    lx = h % LXP;
                } else if (h < 2 * G * LXP) {
                    ly = TY + G + (h - G * LXP) / LXP;
                    lx = (h - G * LXP) % LXP;
                } else {
                    const int r = h - 2 * G * LXP;  // 2G side cells per interior row
                    ly = G + r / (2 * G);
                    const int c2 = r % (2 * G);
                    lx = c2 < G ? c2 : TX + c2;
                }
                halo_lds[j] = ly * LXP + lx;
                halo_xy[j] = lay.at(map_in(ox + lx - G, n0, P.bc), map_in(oy + ly - G, n1, P.bc), 0);
            }
        }
        // the ring of the next plane is loaded while the current plane is
        // computed: raw input (and U0 for the on-the-fly stage) in registers
        double pin[HPT][NV], pu0[HPT][NV];
#pragma unroll
        for (int j = 0; j < HPT; ++j)
#pragma unroll
            for (int v = 0; v < NV; ++v) pin[j][v] = pu0[j][v] = 0.0;
#define AVH_PREFETCH_RING(KP)                                                   \
    _Pragma("unroll") for (int j = 0; j < HPT; ++j) {                           \
        if (has_halo[j]) {                                                      \
            const Idx gi = (Idx)(KP) * lay.plane + halo_xy[j];                  \
            _Pragma("unroll") for (int v = 0; v < NV; ++v) {                    \
                pin[j][v] = ld_in(P, V, v, gi);                                 \
                if (otf) pu0[j][v] = ld_u0(P, V, v, gi);                        \
            }                                                                   \
        }                                                                       \
    }
        AVH_PREFETCH_RING(z0)

        // RK combination ((L*s + U) * ca + U0) * cb (the factor 1 of the RK2
        // stage is exact); U0 of the column's next plane is loaded one plane
        // ahead, with the window's next plane
        const bool combine = !(mode == MODE_FLUX_ONLY || mode == MODE_L);
        const double ca = VOL ? V->ca : (mode == MODE_RK3_2 ? 1. / 3. : (mode == MODE_RK3_3 ? 2.0 : 1.0));
        const double cb = VOL ? V->cb : (mode == MODE_RK2_2 ? 0.5 : (mode == MODE_RK3_2 ? 3. / 4. : 1. / 3.));
        double u0n[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) u0n[v] = 0.0;
        if (combine && col_ok && !ring) {
            const Idx gi = lay.at(ox + cx, oy + cy, z0);
#pragma unroll
            for (int v = 0; v < NV; ++v) u0n[v] = ld_u0(P, V, v, gi);
        }

        for (int k = z0; k < z1; ++k) {
            double* const sp = sp_buf[(k - z0) & 1];
            // plane k into LDS: own column from the window (w[HW-1] is plane k),
            // the halo ring from the prefetched registers
            if (has_col) {
#pragma unroll
                for (int v = 0; v < NV; ++v) sp[v * LP + (cy + G) * LXP + (cx + G)] = w[HW - 1][v];
            }
            bool adm = col_adm;
#pragma unroll
            for (int j = 0; j < HPT; ++j) {
                if (has_halo[j]) {
                    double q[NV];
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        q[v] = pin[j][v];
                        if (otf) q[v] = q[v] * s + pu0[j][v];
                        sp[v * LP + halo_lds[j]] = q[v];
                    }
                    if constexpr (FLUX::FAST) adm = adm & EQ::admitted(q);
                }
            }
            // one vote per wavefront through LDS, read by all after the barrier
            int* const va = s_adm[(k - z0) & 1];
            if constexpr (FLUX::FAST) {
                const bool all = __all(adm);
                if ((threadIdx.x & 63) == 0) va[threadIdx.x >> 6] = all;
            }
            lds_barrier();
            if constexpr (FLUX::FAST) {
                int all = va[0];
#pragma unroll
                for (int i = 1; i < NT / 64; ++i) all = all & va[i];
                adm = all != 0;
            }
            if (k + 1 < z1) {
                AVH_PREFETCH_RING(k + 1)
            }

            double acc[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = 0.0;
            // z: F(k+1/2) from R(k) (kept) and L(k+1) (window centred at k+1)
            double fz[NV], rnext[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) fz[v] = rnext[v] = 0.0;
            // (only for the tile's columns inside the grid: a column past the
            // grid edge supplies the plane's halo but has no cells to update)
            auto z_flux = [&]() {
                // the window's newest plane, here where it is first needed
                if constexpr (FLUX::FAST) {
                    if (has_col) col_adm = col_adm & EQ::admitted(w[WZ - 1]);
                }
                if (col_ok) {
                    typedef typename OpsFor<FLUX::FAST>::type Ops;
                    double lz[NV];
                    bool ok = col_adm;
                    // R(k); a cell itself where nothing is reconstructed
                    const double* const behind = RECON == RECON_NONE ? w[HW - 1] : rprev;
                    recon_faces_reg<RECON, NV, WZ, Ops>(w, HW, rb, lz, rnext);
                    typename EQ::All aL = EQ::template make_all_ops<Ops>(behind, P.gamma, ok);
                    typename EQ::All aR = EQ::template make_all_ops<Ops>(lz, P.gamma, ok);
                    double wz = FLUX::template flux_ops<Ops, 2, EQ>(aL, aR, P.gamma, fz, ok);
                    if (FLUX::FAST && !ok) {
                        // operands outside the guarded range: the plain path
                        recon_face_reg<RECON, NV, false, WZ>(w, HW, lz);
                        recon_face_reg<RECON, NV, true, WZ>(w, HW, rnext);
                        aL = EQ::make_all(behind, P.gamma);
                        aR = EQ::make_all(lz, P.gamma);
                        bool ok2 = true;
                        wz = FLUX::template flux_ops<PlainOps, 2, EQ>(aL, aR, P.gamma, fz, ok2);
                    }
                    ws[2] = ws_max(ws[2], wz);
                }
            };
            auto add_x = [&]() {
                if (has_col) {
                    const int ip = cy * (TX + 1) + cx + 1;
#pragma unroll
                    for (int v = 0; v < NV; ++v)
                        acc[v] = acc[v] + ((-sfx[v * NIMAX + ip]) + sfx[v * NIMAX + ip - 1]);
                }
            };
            auto add_y = [&]() {
                if (has_col) {
                    const int ip = (cy + 1) * TX + cx;
#pragma unroll
                    for (int v = 0; v < NV; ++v)
                        acc[v] = acc[v] + ((-sfy[v * NIMAX + ip]) + sfy[v * NIMAX + ip - TX]);
                }
            };
            // every flux of the plane, then one barrier, then the sums in the
            // reference's x, y, z order
            plane_pass<0>(sp, sfx, ox, oy, P.n, P.gamma, adm, ws[0]);
            plane_pass<1>(sp, sfy, ox, oy, P.n, P.gamma, adm, ws[1]);
            z_flux();
            lds_barrier();
            add_x();
            add_y();
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] = acc[v] + ((-fz[v]) + fprev[v]);

            if (col_ok) {
                const Idx gi = lay.at(ox + cx, oy + cy, k);
                if (ring) {
                    const double* const u0k = slot(k);
#pragma unroll
                    for (int v = 0; v < NV; ++v) u0n[v] = u0k[v * NC];
                }
                double r[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const double l = acc[v];
                    if (!combine) {
                        r[v] = l;
                    } else {
                        double o = l * s;
                        o = o + w[HW - 1][v];
                        o = o * ca;
                        o = o + u0n[v];
                        o = o * cb;
                        r[v] = o;
                    }
                }
                if (final_stage) bad = bad || !EQ::obeys_fast(r, P.gamma);
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    if constexpr (VOL) V->out[v][gi] = r[v];
                    else soa_st<OFF32, false>(P.out, P.ncells, v, gi, r[v]);
                }
                if (mode == MODE_L && P.copy) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) soa_st<OFF32, false>(P.copy, P.ncells, v, gi, w[HW - 1][v]);
                }
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                fprev[v] = fz[v];
                rprev[v] = rnext[v];
            }
            // advance the window to centre k+2
#pragma unroll
            for (int i = 0; i < WZ - 1; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) w[i][v] = w[i + 1][v];
            // the window's next plane and the next write-back's U0, issued
            // together so that their latencies overlap
            if (has_col && k + 1 < z1) {
                const Idx gn = lay.at(gxc, gyc, map_z(k + 2 + HW, n2, P.bc));
                const Idx gw = lay.at(ox + cx, oy + cy, k + 1);
                double cin[NV], cu0[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    cin[v] = ld_in(P, V, v, gn);
                    cu0[v] = 0.0;
                }
                if (otf) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) cu0[v] = ld_u0(P, V, v, gn);
                }
                if (combine && col_ok && !ring) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) u0n[v] = ld_u0(P, V, v, gw);
                }
                if (ring && k + 2 + HW < z1) {
                    double* const kp = slot(k + 2 + HW);
#pragma unroll
                    for (int v = 0; v < NV; ++v) kp[v * NC] = cu0[v];
                }
#pragma unroll
                for (int v = 0; v < NV; ++v) w[WZ - 1][v] = otf ? cin[v] * s + cu0[v] : cin[v];
            }
        }

#undef AVH_PREFETCH_RING
        if (!VOL || mode == MODE_FLUX_ONLY) end_of_tile<NT>(P, ctrl, mode, ws[0], ws[1], ws[2], s_ws, bad, s_end);
    }
};

template <class K>
__global__ __launch_bounds__(256, K::WAVES) void march_kernel3(StageParams P) {
    K::run(P);
}

// A stage over a box of a reference Volume
template <class K>
__global__ __launch_bounds__(256) void volume_march_kernel3(StageParams P, VolumeParams V) {
    K::run(P, &V);
}

}  // namespace avh
