// Whole time steps of a small 1D grid in one launch of one workgroup.
//
// A stage launch of such a grid is all latency: four to five microseconds for
// a few hundred cells, three launches a step.  Here the grid (with its ghost
// cells) stays in the LDS of one workgroup, each thread keeps U0 and the
// current stage's value of its cells in registers, and a stage is two
// barriers: fluxes published, cells published.  The largest wave speed, the
// constraint check and the range check of SharedOps travel as one vote per
// wavefront beside them; the step's bookkeeping (dt, time, save counters, the
// loop test) is evaluated by every thread alike.  The operations and their
// order are those of the stage kernels, so the results have the same bits.
//
// A workgroup takes at most 512 threads and up to four interfaces a thread:
// each wavefront evaluates dt and the bookkeeping for itself, about 200
// instructions a step, and with 1024 threads these were a good part of a step
// (burgers, eno3, 1024 cells: 6.5 us a step with 1024 threads, 4.5 with 512).
// What is left at 200 cells is the chain of one interface's operations, three
// times a step; from 1024 cells on it is the issue rate of the one compute
// unit.  Time of a step, rk3, in microseconds, against stage launches (three,
// or two with avh_pair.hpp):
//   cells              64    200    512   1024   2048
//   burgers none      1.1    1.5    1.9    2.7    4.2
//     three           9.5   10.2   11.2   11.3   11.1
//   burgers weno2     1.9    2.3    3.2    4.9    8.7
//     three, two     11.3   11.3   12.8   12.9   12.7, 9.0
//   euler1 none       3.5    3.9    5.6    9.5
//     three          13.5   13.8   16.2   16.3
//   euler1 eno3       4.5    5.1    7.0   12.4
//     three, two     13.9   14.9   18.3   18.3, 12.8
// so the line lies where the interfaces per thread stop paying: 2048 of them
// for burgers, 1024 for euler1.
#pragma once
#include "avh_stage.hpp"

#pragma clang fp contract(off)

namespace avh {

__host__ __device__ constexpr int line_interfaces(int nv) { return nv == 1 ? 2048 : 1024; }

struct LineParams {
    double* state;  // U0, interior-only SoA
    Control* ctrl;
    int n, bc, integrator;  // 0 forward euler, 1 rk2, 2 rk3
    double gamma;
    int steps;  // at most this many
};

// CPT: cells and interfaces per thread (their number is at most CPT times the
// threads of the launch)
template <class EQ, int RECON, class FLUX, int CPT>
struct LineKernel {
    static constexpr int NV = EQ::NV;
    static constexpr int G = ReconTraits<RECON>::GHOST;
    static constexpr int MAX_THREADS = 512, MAX_WAVES = MAX_THREADS / 64;
    typedef typename OpsFor<FLUX::FAST>::type Ops;

    static size_t lds_bytes(int n) { return sizeof(double) * (size_t)NV * ((n + 2 * G) + (n + 1)); }

    template <class OPS>
    __device__ __forceinline__ static double interface(const double* u, int pitch, int ia, double gamma, double* F,
                                                       bool& ok) {
        double qa[NV], qb[NV];
        recon_face_ops<RECON, NV, true, OPS>(u, pitch, ia, 1, qa);       // right face of cell ia
        recon_face_ops<RECON, NV, false, OPS>(u, pitch, ia + 1, 1, qb);  // left face of the next
        const typename EQ::All aL = EQ::template make_all_ops<OPS>(qa, gamma, ok);
        const typename EQ::All aR = EQ::template make_all_ops<OPS>(qb, gamma, ok);
        return FLUX::template flux_ops<OPS, 0, EQ>(aL, aR, gamma, F, ok);
    }

    static constexpr int UNROLL = 2;
    __device__ static void run(const LineParams& P) {
        extern __shared__ __align__(16) double line_lds[];
        __shared__ double s_ws[MAX_WAVES];
        __shared__ int s_turned[3], s_bad;
        Control* const ctrl = P.ctrl;
        const int n = P.n, pitch = n + 2 * G, nt = blockDim.x;
        const int tid = threadIdx.x, wave = tid >> 6;
        double* const u = line_lds;               // [NV][n + 2G]
        double* const f = line_lds + NV * pitch;  // [NV][n + 1]

        double u0[CPT][NV], us[CPT][NV];
#pragma unroll
        for (int m = 0; m < CPT; ++m)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int c = tid + m * nt;
                u0[m][v] = P.state[(long long)v * n + (c < n ? c : n - 1)];
            }
        StepInputs k = step_inputs(ctrl);
        double t_end = ctrl->t_end;
        long long steps = ctrl->steps;
        int pending = ctrl->saves_pending, violated = ctrl->violated;
        const int pause = ctrl->pause_on_save;
        if (!ctrl->active) return;
        const bool g_ok = EQ::gamma_admitted(P.gamma);

        // cell c's value into LDS, with its boundary images (periodic wrap or
        // neumann mirror of the first and last G cells)
        auto put = [&](int c, const double* q) {
#pragma unroll
            for (int v = 0; v < NV; ++v) u[v * pitch + G + c] = q[v];
            if (c < G) {
                const int at = P.bc == BC_PERIODIC ? n + c : -1 - c;
#pragma unroll
                for (int v = 0; v < NV; ++v) u[v * pitch + G + at] = q[v];
            }
            if (c >= n - G) {
                const int at = P.bc == BC_PERIODIC ? c - n : 2 * n - 1 - c;
#pragma unroll
                for (int v = 0; v < NV; ++v) u[v * pitch + G + at] = q[v];
            }
        };
        // Every thread's cells into LDS and the two votes, for which a wavefront
        // writes only where it has something to say.  Returns, after the
        // barrier, whether all cells are admitted to SharedOps.  Of the three
        // flags one is written and read, and the next is cleared for the
        // following call: its last readers have passed the barrier before.
        // s_bad stays set: the loop ends with the step that set it.
        int slot = 0;
        auto publish = [&](const double (&q)[CPT][NV], bool check) {
            bool adm = g_ok, fail = false;
#pragma unroll
            for (int m = 0; m < CPT; ++m) {
                const int c = tid + m * nt;
                if (c >= n) continue;
                put(c, q[m]);
                if (FLUX::FAST) adm = adm & EQ::admitted(q[m]);
                if (check) fail = fail || !EQ::obeys_fast(q[m], P.gamma);
            }
            const int next = slot == 2 ? 0 : slot + 1;
            if (FLUX::FAST) {
                if (!__all(adm) && (tid & 63) == 0) s_turned[slot] = 1;
                if (tid == 0) s_turned[next] = 0;
            }
            if (check && __any(fail) && (tid & 63) == 0) s_bad = 1;
            lds_barrier();
            const bool all = FLUX::FAST ? s_turned[slot] == 0 : true;
            slot = next;
            return all;
        };
        // fluxes of every interface into f (interface i lies left of cell i;
        // with periodic boundaries the last one is the first)
        const int ni = P.bc == BC_PERIODIC ? n : n + 1;
        auto fluxes = [&](bool adm) {
            double ws = 0.0;
            unsigned int redo = 0;
#pragma unroll UNROLL
            for (int m = 0; m < CPT; ++m) {
                const int i = tid + m * nt;
                if (i >= ni) break;
                double F[NV];
                bool ok = adm;
                const double w = interface<Ops>(u, pitch, G + i - 1, P.gamma, F, ok);
                if (ok) ws = ws_max(ws, w);
                else redo |= 1u << m;
#pragma unroll
                for (int v = 0; v < NV; ++v) f[v * (n + 1) + i] = F[v];
            }
            if (FLUX::FAST && redo != 0) {
                for (int m = 0; m < CPT; ++m) {
                    if (!(redo >> m & 1)) continue;
                    const int i = tid + m * nt;
                    double F[NV];
                    bool ok = true;
                    ws = ws_max(ws, interface<PlainOps>(u, pitch, G + i - 1, P.gamma, F, ok));
#pragma unroll
                    for (int v = 0; v < NV; ++v) f[v * (n + 1) + i] = F[v];
                }
            }
            return ws;
        };
        // net flux of the thread's cells: 0 + ((-F[c+1]) + F[c])
        auto net = [&](int m, double* l) {
            const int c = tid + m * nt < n ? tid + m * nt : n - 1;
            const int r = c + 1 < ni ? c + 1 : 0;
#pragma unroll
            for (int v = 0; v < NV; ++v) l[v] = 0.0 + ((-f[v * (n + 1) + r]) + f[v * (n + 1) + c]);
        };

        if (tid < MAX_WAVES) s_ws[tid] = 0.0;
        if (tid == 0) s_turned[0] = s_bad = 0;
        lds_barrier();
        // one dimension: cells of no size drop out of step_dt
        k.cell[1] = k.cell[2] = 0.0;
        bool adm = publish(u0, false);
        double dt = 0.0;
        int active = 1;
        for (int step = 0; step < P.steps && active; ++step) {
            // first stage: L(U0), the wave speed and dt
            const double w = wave_max63(fluxes(adm));
            if ((tid & 63) == 63) s_ws[wave] = w;
            lds_barrier();
            k.ws[0] = 0.0;
#pragma unroll
            for (int i = 0; i < MAX_WAVES; ++i) k.ws[0] = ws_max(k.ws[0], s_ws[i]);
            dt = step_dt(k);
            const double s = dt / k.cell[0];
#pragma unroll
            for (int m = 0; m < CPT; ++m) {
                double l[NV];
                net(m, l);
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    double o = l[v] * s;
                    o = o + u0[m][v];
                    us[m][v] = o;
                }
            }
            adm = publish(us, P.integrator == 0);
            for (int st = 1; st <= P.integrator; ++st) {
                fluxes(adm);
                lds_barrier();
                // rk2: ((L*s + U1) + U0) * 0.5; rk3: ((L*s + U1)*(1/3) + U0)*(3/4),
                // then ((L*s + U2)*2 + U0)*(1/3)
                const double ca = P.integrator == 1 ? 1.0 : (st == 1 ? 1. / 3. : 2.0);
                const double cb = P.integrator == 1 ? 0.5 : (st == 1 ? 3. / 4. : 1. / 3.);
#pragma unroll
                for (int m = 0; m < CPT; ++m) {
                    double l[NV];
                    net(m, l);
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        double o = l[v] * s;
                        o = o + us[m][v];
                        o = o * ca;
                        o = o + u0[m][v];
                        o = o * cb;
                        us[m][v] = o;
                    }
                }
                adm = publish(us, st == P.integrator);
            }
#pragma unroll
            for (int m = 0; m < CPT; ++m)
#pragma unroll
                for (int v = 0; v < NV; ++v) u0[m][v] = us[m][v];
            // end of the step, as end_step
            k.t = k.t + dt;
            ++steps;
            if (s_bad) {
                violated = 1;
            } else {
#pragma unroll
                for (int i = 0; i < MAX_ADJ; ++i)
                    if (i < k.n_adj && k.t >= (double)k.saved[i] * k.interval[i] + k.start[i]) {
                        k.saved[i] = k.saved[i] + 1;
                        ++pending;
                    }
            }
            active = (!(k.t >= t_end) && !violated && !(pause && pending > 0)) ? 1 : 0;
        }

#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int c = tid + m * nt;
            if (c >= n) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) P.state[(long long)v * n + c] = u0[m][v];
        }
        if (tid == 0) {
            ctrl->dt = dt;
            ctrl->scale = dt / k.cell[0];
            ctrl->t = k.t;
            ctrl->steps = steps;
            ctrl->last_dt = dt;
            if (violated) ctrl->violated = 1;
#pragma unroll
            for (int i = 0; i < MAX_ADJ; ++i) ctrl->adj_saved[i] = k.saved[i];
            ctrl->saves_pending = pending;
            ctrl->block_violation = 0;
            clear_wave_speeds(ctrl);
            ctrl->active = active;
        }
    }
};

template <class K>
__global__ __launch_bounds__(K::MAX_THREADS) void line_kernel(LineParams P) {
    K::run(P);
}

}  // namespace avh
