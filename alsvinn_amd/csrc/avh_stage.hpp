// Fused FP64 finite-volume stage kernels: what all of them share, and the 1D
// one (2D: avh_stage2d.hpp, 3D: avh_stage3d.hpp).
//
// One launch = one RK stage over the whole grid.  Each workgroup owns a tile
// of interior cells:
//   1. stage the tile plus a GHOST-wide halo of the stage input into LDS;
//      halo cells outside the domain are read through the boundary map
//      (periodic wrap / neumann mirror), which is the ghost fill of the
//      reference done at load time; in the on-the-fly modes the stage input
//      is formed while loading as U1 = L0*s + U0;
//   2. per direction: every interface, reconstructing the right face of the
//      left cell and the left face of the right cell and evaluating the
//      numerical flux; fluxes go to LDS, the interface wave speeds to a
//      per-thread max;
//   3. each thread accumulates the net flux of its cells in registers,
//      out = 0 + ((-F[i+1/2]) + F[i-1/2]) per direction, exactly as
//      NumericalFluxCPU::computeNetFlux does on a zeroed output;
//   4. the RK stage combination of the integrator, the constraint check of
//      the final stage, and the write of the result.
// The CFL wave speed is reduced with DPP moves within a wavefront and one
// atomicMax per direction per workgroup (non-negative doubles order like their
// bit patterns); the launches after the first stage derive dt from those maxima
// themselves, and the last workgroup of the last one ends the step (time, save
// counters, loop test), so a whole time step runs without a host round trip and
// without grid-wide fences.  Forward euler, whose last pass is element-wise, and
// batches end theirs in a launch of one workgroup.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "avh_physics.hpp"

#pragma clang fp contract(off)

namespace avh {

constexpr int MAX_ADJ = 4;

// Device-resident step bookkeeping.  Written by the host between launches,
// by atomics (wave-speed maxima, violation flag) and by finish_step_kernel.
struct Control {
    unsigned long long ws_bits[3];  // running max wave speed per direction (double bits)
    double t;                        // current time (TimestepInformation)
    double dt;                       // dt of the step in flight
    double scale;                    // dt / dx (RungeKutta*: output *= dt/cellLengths.x)
    double last_dt;
    double t_end;
    double cfl;
    double cell[3];
    double adj_interval[MAX_ADJ];
    double adj_start[MAX_ADJ];
    long long adj_saved[MAX_ADJ];  // FixedIntervalWriter::numberSaved
    long long steps;
    int n_adj;
    int active;         // 1 while the step in flight must run
    int violated;       // sticky constraint failure
    int saves_pending;  // fixed-interval save times reached, not yet acknowledged
    int pause_on_save;
    int block_violation;
    // workgroups of a finishing stage launch that are done (low 32 bits) and
    // how many of them found a constraint violation (high 32 bits); the last
    // one runs the end of the step and sets it back to 0
    unsigned long long arrive;
};

enum StageMode {
    MODE_FLUX_ONLY = 0,  // out = net flux, wave speeds accumulated, nothing else
    MODE_L = 1,          // first stage: out = L(U0), last block computes dt
    MODE_RK2_2 = 2,      // in = L0*s+U0; out = ((L*s + U1) + U0) * 0.5, ends step
    MODE_RK3_2 = 3,      // in = L0*s+U0; out = ((L*s + U1) * (1/3) + U0) * (3/4)
    MODE_RK3_3 = 4       // in = U2;      out = ((L*s + U2) * 2 + U0) * (1/3), ends step
};

// modes whose input is U1 = L0*s + U0, formed as the tile loads
__host__ __device__ __forceinline__ constexpr bool on_the_fly(int mode) {
    return mode == MODE_RK3_2 || mode == MODE_RK2_2;
}

enum { BC_PERIODIC = 0, BC_NEUMANN = 1 };

struct StageParams {
    const double* in;  // stage input U_s, or L0 in the on-the-fly modes
    const double* u0;  // U0 (on-the-fly input and RK combination)
    double* out;       // stage output (may equal u0 in MODE_RK3_3:
                       // u0 is then read only at the cell being written)
    Control* ctrl;
    long long ncells;  // interior cells; variable stride of every buffer
    int n[3];
    int bc;
    int mode;
    double gamma;
    // 1: the launch is the step's last stage and its last workgroup runs the
    // end of the step (end_step); 0: the caller runs finish_step_kernel
    int finish = 0;
    // MODE_L: where each cell's input is written as well, unless null.  RK2's
    // second stage overwrites the state, and reads neighbours' U0 from here, to
    // form U1 = L0*s + U0 as it loads: an element-wise pass for U1 took 6.6 of a
    // 501x333 step's 46 us, the copy and the second operand together 2.
    double* copy = nullptr;
    int lz = 0;  // 3D: planes a workgroup marches through (set by the launcher)
};

// The reference's Volume (alsfvm/src/volume/Volume.cpp:44-60): one array per
// conserved variable including its ghost cells, x fastest.  A stage kernel
// instantiated for it covers a box of the interior (P.n = the box's extent)
// and reads the halo from the ghost cells exactly as the caller filled them
// (boundary conditions or a neighbour's cells), as the reference's
// NumericalFlux::computeFlux does.
struct VolumeParams {
    const double* in[5];
    double* out[5];
    int tot[3];    // cells per axis including ghosts
    int ghost[3];  // ghost cells per axis of the volume
    int org[3];    // first cell of the box, interior coordinates
    // a combination in place of the net flux L: out = ((L*s + in) * ca + u0) * cb
    const double* u0[5];
    double s, ca, cb;
};

__device__ __forceinline__ long long volume_index(const VolumeParams& V, int x, int y, int z) {
    return ((long long)(z + V.org[2] + V.ghost[2]) * V.tot[1] + (y + V.org[1] + V.ghost[1])) * V.tot[0] +
           (x + V.org[0] + V.ghost[0]);
}

// Element v of cell gi of an SoA buffer of nc cells per variable.  With
// OFF32 the cell index is a 32-bit value (the caller guarantees nc < 2^29,
// so byte offsets stay below 2^32) and the variable's base a uniform value
// the compiler cannot re-associate with the lane offset: the access is then
// a global load / store with a scalar base and a 32-bit lane offset, with no
// 64-bit address arithmetic per lane.
typedef __attribute__((address_space(1))) char global_char;
__device__ __forceinline__ global_char* uniform_base(const double* p) {
    const unsigned long long a = (unsigned long long)p;
    const unsigned int lo = __builtin_amdgcn_readfirstlane((unsigned int)a);
    const unsigned int hi = __builtin_amdgcn_readfirstlane((unsigned int)(a >> 32));
    return (global_char*)(((unsigned long long)hi << 32) | lo);
}
template <bool OFF32, class Idx>
__device__ __forceinline__ double soa_ld(const double* base, long long nc, int v, Idx gi) {
    if constexpr (OFF32) {
        return *(const __attribute__((address_space(1))) double*)(uniform_base(base + v * nc) + gi * 8u);
    } else {
        return base[v * nc + gi];
    }
}
// The 1D and 2D kernels store their results through the L2 (agent scope: each
// XCD has an L2 of its own, so such a store goes on to memory).  A kernel's end
// otherwise writes back what the L2s hold dirty, up to 32 MB, before the next
// launch may start.  Step time, us: 501x333 rk3 39.9 -> 38.3, eno3 rk2 31.2 ->
// 29.9, 256^2 26.2 -> 25.7, 1024^2 125.1 -> 123.8.  The 3D march stores
// plainly (through the L2 256^3 is 0.9 % slower, 97x83x61 1 %, a volume substep
// at 128^3 2.6 %: its stores are partial lines that the L2 merges).
template <class Ptr>
__device__ __forceinline__ void store_through(Ptr p, double x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool OFF32, bool THROUGH, class Idx>
__device__ __forceinline__ void soa_st(double* base, long long nc, int v, Idx gi, double x) {
    if constexpr (OFF32) {
        const auto p = (__attribute__((address_space(1))) double*)(uniform_base(base + v * nc) + gi * 8u);
        if constexpr (THROUGH) store_through(p, x);
        else *p = x;
    } else {
        if constexpr (THROUGH) store_through(base + v * nc + gi, x);
        else base[v * nc + gi] = x;
    }
}

// Boundary map of a coordinate in [-G, n+G) onto the interior: periodic wrap
// (alsfvm/include/alsfvm/boundary/Periodic.hpp:24-42) or neumann mirror
// (alsfvm/include/alsfvm/boundary/Neumann.hpp:24-35).  Applied per axis this
// reproduces the reference's x -> y -> z fill order, corners included.
__device__ __forceinline__ int bc_map(int g, int n, int bc) {
    if (g < 0) return bc == BC_PERIODIC ? g + n : -1 - g;
    if (g >= n) return bc == BC_PERIODIC ? g - n : 2 * n - 1 - g;
    return g;
}

__device__ __forceinline__ double ws_max(double acc, double v) {
    // std::max(acc, v): NaN candidates leave acc unchanged
    return (acc < v) ? v : acc;
}

// The largest of a wavefront's values, none negative or NaN, in lane 63: within
// rows of 16 lanes, then rows of 32 and 64, by DPP moves (lanes without a
// partner see 0).  Shuffles go through LDS and took 0.2 us of a 200-cell step.
template <int CTRL>
__device__ __forceinline__ double dpp_max(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned int lo = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)(unsigned int)b, CTRL, 0xf, 0xf, false);
    const unsigned int hi = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)(unsigned int)(b >> 32), CTRL, 0xf, 0xf, false);
    return fmax(v, __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo)));
}
__device__ __forceinline__ double wave_max63(double v) {
    v = dpp_max<0x111>(v);  // row_shr:1, 2, 4, 8
    v = dpp_max<0x112>(v);
    v = dpp_max<0x114>(v);
    v = dpp_max<0x118>(v);
    v = dpp_max<0x142>(v);  // row_bcast:15, 31
    return dpp_max<0x143>(v);
}

__device__ __forceinline__ unsigned int tile_id_xcd(unsigned int b, unsigned int nb) {
    // Workgroups are dealt to the 8 XCDs round-robin; give each XCD a
    // contiguous run of tiles so tiles sharing halos share an L2.
    const unsigned int nfull = nb - nb % 8u;
    if (b >= nfull) return b;
    return (b % 8u) * (nfull / 8u) + b / 8u;
}

// largest wave speed recorded along direction d
__host__ __device__ __forceinline__ double wave_speed(const Control* c, int d) {
    double w;
    __builtin_memcpy(&w, &c->ws_bits[d], sizeof w);
    return w;
}

__host__ __device__ __forceinline__ void clear_wave_speeds(Control* c) {
    for (int d = 0; d < 3; ++d) c->ws_bits[d] = 0ull;
}

// dt of the step in flight: cfl / sum_d(ws_d / dx_d), then the
// FixedIntervalWriter clips (alsfvm/src/integrator/Integrator.cpp:20-66,
// alsfvm/src/io/FixedIntervalWriter.cpp:45-53).  ws_d are the maxima the
// first stage accumulated; every launch after it evaluates this same
// expression, so all of them use the identical dt without a grid-wide
// barrier or fence.
// Everything it reads is loaded before anything is used: the loads then cost
// one latency, which on small grids is a good part of a launch.
struct StepInputs {
    double ws[3], cell[3], cfl, t;
    double interval[MAX_ADJ], start[MAX_ADJ];
    long long saved[MAX_ADJ];
    int n_adj;
};
__device__ __forceinline__ StepInputs step_inputs(const Control* c) {
    StepInputs k;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        k.ws[d] = wave_speed(c, d);
        k.cell[d] = c->cell[d];
    }
    k.cfl = c->cfl;
    k.t = c->t;
    k.n_adj = c->n_adj;
#pragma unroll
    for (int i = 0; i < MAX_ADJ; ++i) {
        k.interval[i] = c->adj_interval[i];
        k.start[i] = c->adj_start[i];
        k.saved[i] = c->adj_saved[i];
    }
    return k;
}
__device__ __forceinline__ double step_dt(const StepInputs& k) {
    double total = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (k.cell[d] == 0) continue;
        total += k.ws[d] / k.cell[d];
    }
    double dt = k.cfl / total;
#pragma unroll
    for (int i = 0; i < MAX_ADJ; ++i) {
        if (i < k.n_adj && k.saved[i] > 0) {
            const double next = (double)k.saved[i] * k.interval[i] + k.start[i];
            const double cand = next - k.t;
            dt = (cand < dt) ? cand : dt;
        }
    }
    return dt;
}
__device__ __forceinline__ double step_dt(const Control* c) { return step_dt(step_inputs(c)); }

// End of a step: t += dt, constraint flag, then the writers' save counters
// (alsfvm/src/simulator/Simulator.cpp:81-85, 180-214;
// alsfvm/src/io/FixedIntervalWriter.cpp:33-43) and the loop test
// `t >= endTime` (Simulator.cpp:77-79); clears the wave-speed maxima for the
// next step.  Nothing in it but the constraint flag depends on the launch that
// ends the step, so it is worked out (StepEnd) by a thread of every workgroup
// while the workgroup's loads are in flight, and the last one to finish only
// writes it (a 64^2 step: 14.2 -> 13.9 us, 128^2 17.0 -> 16.5).
struct EndInputs {
    double t_end;
    long long steps;
    int violated, pause, pending;
};
__device__ __forceinline__ EndInputs end_inputs(const Control* c) {
    return EndInputs{c->t_end, c->steps, c->violated, c->pause_on_save, c->saves_pending};
}
struct StepEnd {
    double t, dt, scale;
    long long steps, saved[MAX_ADJ];
    int pending, more;  // without a violation
};
__device__ __forceinline__ void prepare_end(const StepInputs& k, const EndInputs& e, double dt, StepEnd* r) {
    const double t = k.t + dt;
    int pending = e.pending;
#pragma unroll
    for (int i = 0; i < MAX_ADJ; ++i) {
        const bool save = i < k.n_adj && t >= (double)k.saved[i] * k.interval[i] + k.start[i];
        r->saved[i] = k.saved[i] + (save ? 1 : 0);
        pending += save ? 1 : 0;
    }
    r->t = t;
    r->dt = dt;
    r->scale = dt / k.cell[0];
    r->steps = e.steps + 1;
    r->pending = pending;
    r->more = (!(t >= e.t_end) && !e.violated && !(e.pause && pending > 0)) ? 1 : 0;
}
__device__ __forceinline__ void end_step(Control* c, const StepEnd& r, bool violation) {
    c->dt = r.dt;
    c->scale = r.scale;
    c->t = r.t;
    c->steps = r.steps;
    c->last_dt = r.dt;
    if (violation) {
        c->violated = 1;
    } else {
#pragma unroll
        for (int i = 0; i < MAX_ADJ; ++i) c->adj_saved[i] = r.saved[i];
        c->saves_pending = r.pending;
    }
    c->block_violation = 0;
    clear_wave_speeds(c);
    c->active = !violation && r.more ? 1 : 0;
}

// Thread 0 of every workgroup of a step's last stage reports here once the
// workgroup's cells are written (`bad`: a cell broke the constraints); the
// last workgroup to arrive ends the step.  The count and the violations
// travel in one atomic, so no fence is needed: the end of the step holds only
// what earlier launches wrote (the first stage's wave speeds, the previous
// step's bookkeeping).
__device__ __forceinline__ void arrive_final(Control* c, const StepEnd& r, bool bad) {
    const unsigned long long add = 1ull + (bad ? (1ull << 32) : 0ull);
    const unsigned long long prev = atomicAdd(&c->arrive, add);
    if ((unsigned int)prev == gridDim.x - 1) {
        c->arrive = 0ull;
        end_step(c, r, ((prev + add) >> 32) != 0ull);
    }
}

// dt / dx of the step in flight; where this launch ends the step, thread 0
// also works out its end.
__device__ __forceinline__ double stage_scale(const StageParams& P, const Control* c, int mode, StepEnd* r) {
    const StepInputs k = step_inputs(c);
    const bool ends = (mode == MODE_RK2_2 || mode == MODE_RK3_3) && P.finish;
    EndInputs e{};
    if (ends) e = end_inputs(c);
    const double dt = step_dt(k);
    if (ends && threadIdx.x == 0) prepare_end(k, e, dt, r);
    return dt / k.cell[0];
}

// What a workgroup leaves behind after its cells.  First stage and flux-only:
// the wave speeds, a wavefront reduction, then one atomicMax per direction
// (non-negative doubles order like their bit patterns).  Final stage: whether
// a cell broke the constraints, and the end of the step.
template <int NT>
__device__ __forceinline__ void end_of_tile(const StageParams& P, Control* ctrl, int mode, double w0, double w1,
                                            double w2, double (*s_ws)[NT / 64], bool bad, const StepEnd& end) {
    if (mode == MODE_FLUX_ONLY || mode == MODE_L) {
        const double ws[3] = {w0, w1, w2};
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double w = wave_max63(ws[d]);
            if (lane == 63) s_ws[d][wid] = w;
        }
        lds_barrier();
        if (threadIdx.x < 3) {
            double w = 0.0;
#pragma unroll
            for (int i = 0; i < NT / 64; ++i) w = ws_max(w, s_ws[threadIdx.x][i]);
            if (w > 0.0) atomicMax(&ctrl->ws_bits[threadIdx.x], (unsigned long long)__double_as_longlong(w));
        }
    } else if (mode == MODE_RK2_2 || mode == MODE_RK3_3) {
        const int any_bad = __syncthreads_or(bad);
        if (threadIdx.x == 0) {
            if (P.finish) arrive_final(ctrl, end, any_bad != 0);
            else if (any_bad) atomicOr(&ctrl->block_violation, 1);
        }
    }
}

// 1D grids too large for one workgroup (avh_line.hpp): a tile of TX cells.
template <class EQ, int RECON, class FLUX, int TX, int NT>
struct StageKernel1 {
    typedef typename OpsFor<FLUX::FAST>::type Ops;
    static constexpr int NV = EQ::NV;
    static constexpr int G = ReconTraits<RECON>::GHOST;
    static constexpr int LT = TX + 2 * G;  // tile cells incl. halo
    static constexpr int NI = TX + 1;
    static constexpr int NTHREADS = NT;
    static constexpr int CPT = (TX + NT - 1) / NT;  // cells per thread

    // reconstruct both sides of the interface between cells ia and ia + 1 (LDS
    // indices) and evaluate the numerical flux under OPS; `ok` comes in as
    // whether the cells are admitted to SharedOps
    template <class OPS>
    __device__ __forceinline__ static double interface(const double* su, int ia, double gamma, double* F, bool& ok) {
        double qa[NV], qb[NV];
        recon_face_ops<RECON, NV, true, OPS>(su, LT, ia, 1, qa);       // right face of a
        recon_face_ops<RECON, NV, false, OPS>(su, LT, ia + 1, 1, qb);  // left face of b
        const typename EQ::All aL = EQ::template make_all_ops<OPS>(qa, gamma, ok);
        const typename EQ::All aR = EQ::template make_all_ops<OPS>(qb, gamma, ok);
        return FLUX::template flux_ops<OPS, 0, EQ>(aL, aR, gamma, F, ok);
    }

    __device__ static void run(const StageParams& P) { run_tile(P, tile_id_xcd(blockIdx.x, gridDim.x)); }
    __device__ static void run_volume(const StageParams& P, const VolumeParams& V) {
        run_tile<true>(P, tile_id_xcd(blockIdx.x, gridDim.x), &V);
    }

    // number of tiles covering a grid of n cells
    __host__ __device__ static unsigned int tiles(const int* n) { return (unsigned int)((n[0] + TX - 1) / TX); }

    // VOL: the cells live in a reference Volume (V; MODE_FLUX_ONLY, or
    // MODE_RK3_3 for the combination V describes) and P.n is the extent of the
    // box the launch covers; otherwise in the interior-only buffers of P with
    // the boundary map for the halo.
    template <bool VOL = false>
    __device__ static void run_tile(const StageParams& P, const unsigned int tile, const VolumeParams* V = nullptr) {
        __shared__ double su[NV * LT];
        __shared__ double sf[NV * NI];
        __shared__ double s_ws[3][NT / 64];
        __shared__ StepEnd s_end;
        __shared__ int s_adm[NT / 64];

        Control* ctrl = P.ctrl;
        const int mode = P.mode;
        if (!VOL && !ctrl->active && mode != MODE_FLUX_ONLY) return;  // step past the end: no-op

        const int n0 = P.n[0];
        const int ox = (int)tile * TX;
        const long long nc = P.ncells;
        const bool otf = on_the_fly(mode);
        const double s = (mode == MODE_FLUX_ONLY || mode == MODE_L) ? 0.0
                         : VOL                                       ? V->s
                                                                     : stage_scale(P, ctrl, mode, &s_end);

        // 1. stage input tile + halo into LDS through the boundary map.  Each
        // thread issues the loads of all its points before writing any of
        // them, so that their global-memory latencies overlap; points past
        // the tile repeat the last one and are not written.
        constexpr int SPT = (LT + NT - 1) / NT;  // staged points per thread
        long long sg[SPT];
#pragma unroll
        for (int k = 0; k < SPT; ++k) {
            int p = threadIdx.x + k * NT;
            p = p < LT ? p : LT - 1;
            int gx = ox + p - G;
            gx = gx < n0 + G ? gx : n0 + G - 1;
            if constexpr (VOL) sg[k] = volume_index(*V, gx, 0, 0);
            else sg[k] = bc_map(gx, n0, P.bc);
        }
        double sv[SPT][NV];
#pragma unroll
        for (int k = 0; k < SPT; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                if constexpr (VOL) sv[k][v] = V->in[v][sg[k]];
                else sv[k][v] = P.in[v * nc + sg[k]];
            }
        if (otf) {
#pragma unroll
            for (int k = 0; k < SPT; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) sv[k][v] = sv[k][v] * s + P.u0[v * nc + sg[k]];
        }
#pragma unroll
        for (int k = 0; k < SPT; ++k) {
            const int p = threadIdx.x + k * NT;
            if (LT % NT != 0 && p >= LT) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) su[v * LT + p] = sv[k][v];
        }
        // whether SharedOps may run on this tile: one vote per wavefront
        // through LDS, read by all after the barrier that publishes the tile
        bool adm = EQ::gamma_admitted(P.gamma);
        if constexpr (FLUX::FAST) {
#pragma unroll
            for (int k = 0; k < SPT; ++k) adm = adm & EQ::admitted(sv[k]);
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

        // 2. interface fluxes into LDS; interface i lies right of cell i - 1.
        // A FAST flux evaluates each with SharedOps, and with PlainOps where
        // the operands leave the range in which SharedOps is exact.
        double ws = 0.0;
        for (int it = threadIdx.x; it < NI; it += NT) {
            if (ox + it - 1 >= n0) continue;
            double F[NV];
            bool ok = adm;
            double w = interface<Ops>(su, it - 1 + G, P.gamma, F, ok);
            if (FLUX::FAST && !ok) {
                ok = true;
                w = interface<PlainOps>(su, it - 1 + G, P.gamma, F, ok);
            }
            ws = ws_max(ws, w);
#pragma unroll
            for (int v = 0; v < NV; ++v) sf[v * NI + it] = F[v];
        }
        lds_barrier();

        // 3. net flux, RK combination and write-back; the U0 loads of all the
        // thread's cells are issued first (cells outside the grid load element
        // 0 and write nothing)
        bool bad = false;
        const bool final_stage = !VOL && (mode == MODE_RK2_2 || mode == MODE_RK3_3);
        const bool combine = !(mode == MODE_FLUX_ONLY || mode == MODE_L);
        long long gc[CPT];
        bool inside[CPT];
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = threadIdx.x + m * NT;
            inside[m] = (TX % NT == 0 || c < TX) && ox + c < n0;
            if constexpr (VOL) gc[m] = inside[m] ? volume_index(*V, ox + c, 0, 0) : 0;
            else gc[m] = inside[m] ? ox + c : 0;
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
                    else u0c[m][v] = P.u0[v * nc + gc[m]];
                }
        }
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            if (!inside[m]) continue;
            const int c = threadIdx.x + m * NT;
            double r[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                // temp = -F; out[i] = 0 + (temp[i] + (-1)*temp[i-1])
                const double l = 0.0 + ((-sf[v * NI + c + 1]) + sf[v * NI + c]);
                if (!combine) {
                    r[v] = l;
                } else {
                    // ((L*s + U) * ca + U0) * cb; the factor 1 of the RK2
                    // stage is exact, so every mode keeps its own rounding
                    double o = l * s;
                    o = o + su[v * LT + c + G];
                    o = o * ca;
                    o = o + u0c[m][v];
                    o = o * cb;
                    r[v] = o;
                }
            }
            if (final_stage) bad = bad || !EQ::obeys_fast(r, P.gamma);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                store_through(VOL ? V->out[v] + gc[m] : P.out + v * nc + gc[m], r[v]);
            }
            if (mode == MODE_L && P.copy) {
#pragma unroll
                for (int v = 0; v < NV; ++v) store_through(P.copy + v * nc + gc[m], su[v * LT + c + G]);
            }
        }
        if (!VOL || mode == MODE_FLUX_ONLY) end_of_tile<NT>(P, ctrl, mode, ws, 0.0, 0.0, s_ws, bad, s_end);
    }
};

template <class K>
__global__ __launch_bounds__(K::NTHREADS) __attribute__((amdgpu_waves_per_eu(4))) void stage_kernel(StageParams P) {
    K::run(P);
}

// A stage over a box of a reference Volume
template <class K>
__global__ __launch_bounds__(256) void volume_stage_kernel(StageParams P, VolumeParams V) {
    K::run_volume(P, V);
}

}  // namespace avh
