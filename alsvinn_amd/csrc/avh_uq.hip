// Batched Monte Carlo UQ on the hip platform: sample generation (the
// reference's STLMersenne + Uniform), batched solver groups, end-of-step
// bookkeeping and on-device Welford statistics (C ABI in alsvinn_hip.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <limits>
#include <mutex>
#include <new>
#include <random>
#include <vector>

#include "avh_internal.hpp"

#pragma clang fp contract(off)

using namespace avh;

namespace avh {

// One block per group: every sample's end of step, then a stable (sample
// order) compaction of the samples that reached a statistics save, each with
// its Welford count.
__global__ __launch_bounds__(1024) void batch_finish_kernel(StatsParams S) {
    __shared__ int s_wave[16];
    __shared__ int s_base;
    __shared__ int s_active;
    const StatsGroup& G = S.g[blockIdx.x];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    if (threadIdx.x == 0) {
        s_base = 0;
        s_active = 0;
    }
    __syncthreads();
    for (int base = 0; base < G.nsamples; base += blockDim.x) {
        const int s = base + threadIdx.x;
        int hit = -1;
        if (s < G.nsamples) {
            hit = finish_sample(G.ctrl + s, S.stats_adj);
            if (hit >= 0) hit -= S.save_offset;
            if (G.ctrl[s].active) atomicAdd(&s_active, 1);
        }
        const bool flag = hit >= 0;
        const unsigned long long ball = __ballot(flag);
        const int before = __popcll(ball & ((1ull << lane) - 1ull));
        if (lane == 0) s_wave[wid] = __popcll(ball);
        __syncthreads();
        int off = s_base;
        for (int w = 0; w < wid; ++w) off += s_wave[w];
        if (flag) {
            G.list[3 * (off + before) + 0] = s;
            G.list[3 * (off + before) + 1] = hit;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int tot = 0;
            for (int w = 0; w < nw; ++w) tot += s_wave[w];
            s_base += tot;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        // Welford counts, in list order
        for (int j = 0; j < s_base; ++j) {
            const int k = G.list[3 * j + 1];
            const long long nk = (k < G.nsaves) ? ++G.counts[k] : 0;
            G.list[3 * j + 2] = (int)nk;
        }
        *G.list_len = s_base;
        *G.active_count = s_active;
        __hip_atomic_store(G.host_active, s_active, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}


// Statistics of the initial state (writeInitialTimestep): every sample at
// save index 0, in sample order.
__global__ __launch_bounds__(256) void batch_initial_save_kernel(StatsParams S) {
    const StatsGroup& G = S.g[blockIdx.x];
    for (int s = threadIdx.x; s < G.nsamples; s += blockDim.x) {
        G.list[3 * s + 0] = s;
        G.list[3 * s + 1] = 0;
        G.list[3 * s + 2] = s + 1;
        if (S.stats_adj >= 0) G.ctrl[s].adj_saved[S.stats_adj] = 1;
    }
    if (threadIdx.x == 0) {
        *G.list_len = G.nsamples;
        if (G.nsaves > 0) G.counts[0] = G.nsamples;
    }
}

// 2D Kelvin-Helmholtz fill from per-sample band interfaces lo[x] < y < hi[x]
// at cell midpoints: rho = 2, ux = -0.5 inside, rho = 1, ux = 0.5 outside,
// uy = 0, p = 2.5; conserved with m = u*rho, E = p/(gamma-1) + 0.5*rho*(u.u)
// (alsfvm/include/alsfvm/equation/euler/Euler.hpp:236-245).
__global__ __launch_bounds__(256) void kh2d_fill_kernel(double* state, long long stride, int nx, int ny,
                                                        const double* iface, int nsamples, double lower_y,
                                                        double dy, double gamma) {
    const long long nc = (long long)nx * ny;
    const long long total = nc * nsamples;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (long long)gridDim.x * blockDim.x) {
        const int s = (int)(t / nc);
        const long long i = t % nc;
        const int x = (int)(i % nx), y = (int)(i / nx);
        const double ym = lower_y + dy * y + dy / 2.0;
        const double lo = iface[(long long)s * 2 * nx + x];
        const double hi = iface[(long long)s * 2 * nx + nx + x];
        const bool band = (ym > lo) && (ym < hi);
        const double rho = band ? 2.0 : 1.0;
        const double ux = band ? -0.5 : 0.5;
        const double uy = 0.0;
        const double p = 2.5;
        double dot = ux * ux;
        dot = dot + uy * uy;
        double* q = state + (long long)s * stride;
        q[i] = rho;
        q[nc + i] = ux * rho;
        q[2 * nc + i] = uy * rho;
        q[3 * nc + i] = p / (gamma - 1) + 0.5 * rho * dot;
    }
}


// Sum over the 256 threads of a workgroup, the same tree every time: lanes of
// a wavefront, then the four wavefronts.  The total is thread 0's.
__device__ __forceinline__ double block_sum(double v) {
    __shared__ double s_part[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
    __syncthreads();
    return (s_part[0] + s_part[1]) + (s_part[2] + s_part[3]);
}

// Kinetic energy of one velocity component per sample,
//   E_c = (sum over cells of 0.5 * rho * u_c * u_c) * dV,  u_c = m_c / rho,
// a functional of the conserved state modelled on the Moment functional
// (alsfvm/src/functional/Moment.cpp:31-45).  Block (x, y) sums cells
// x * 256, ... of every gridDim.x-th 256 of sample y; sums_finish_kernel adds
// the blocks' sums in block order, so the result does not depend on timing.  One
// block alone scales its sum itself (a launch less: 100 samples of 200 cells
// 26.7 -> 25.1 us).
// Bound by reading two of the state's variables; one block a sample left all
// but a few CUs idle (16 samples of 256^2: 85 us, now 7 us in 32 blocks each).
__global__ __launch_bounds__(256) void kinetic_energy_kernel(const double* state, long long stride, long long ncells,
                                                             int comp, double scale, double* partial) {
    const double* q = state + (long long)blockIdx.y * stride;
    double acc = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < ncells; i += (long long)gridDim.x * 256) {
        const double rho = q[i];
        const double u = q[(long long)(1 + comp) * ncells + i] / rho;
        acc = acc + 0.5 * rho * (u * u);
    }
    const double sum = block_sum(acc);
    if (threadIdx.x == 0)
        partial[(long long)blockIdx.y * gridDim.x + blockIdx.x] = gridDim.x == 1 ? scale * sum : sum;
}

// out[t] = scale * (sum of the n partials of t), one wavefront each
__global__ __launch_bounds__(256) void sums_finish_kernel(const double* partial, int n, int count, double scale,
                                                          double* out) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (t >= count) return;
    const double* q = partial + (long long)t * n;
    double acc = 0.0;
    for (int k = lane; k < n; k += 64) acc = acc + q[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc = acc + __shfl_xor(acc, off, 64);
    if (lane == 0) out[t] = scale * acc;
}

template <int P>
__device__ __forceinline__ double fast_power(double x) {
    if constexpr (P == 1) {
        return x;
    } else {
        return x * fast_power<P - 1>(x);
    }
}

// acc + |d|^P (P = 0: any power p)
template <int P>
__device__ __forceinline__ double add_power(double acc, double d, double p) {
    if constexpr (P == 2) {
        return fma(d, d, acc);
    } else if constexpr (P > 0) {
        return acc + fast_power<P>(fabs(d));
    } else {
        return acc + pow(fabs(d), p);
    }
}

__device__ __forceinline__ int bc_value_index(int x, int n, int bc) {
    // ValueAtBoundary: periodic wraps, neumann clamps to the interior
    // (alsfvm/include/alsfvm/boundary/ValueAtBoundary.hpp)
    if (bc == AVH_BC_PERIODIC) {
        x %= n;
        return x < 0 ? x + n : x;
    }
    return x < 0 ? 0 : (x > n - 1 ? n - 1 : x);
}

// Structure function of one variable per sample (the structure_cube
// statistic, alsfvm/include/alsfvm/functional/structure_common.hpp:36-154):
// for every cell and lag h, |u - u'|^p summed over the cells u' on the
// boundary of the square of half-width h around it (2 points in 1D, 8h in
// 2D), divided by the number of cells.
//
// One thread a cell: block (x, y, z) sums 256 cells of sample z at lag y + 1.
// With periodic boundaries of a 2D grid one side of the ring is summed (see the
// sweep below).  Serves 1D grids, and 2D ones as structure_sweeps says.
template <int P>
__global__ __launch_bounds__(256) void structure_gather_kernel(const double* state, long long stride, int var, int nx,
                                                               int ny, int dims, int bc, double p, double* partial) {
    const int h = blockIdx.y + 1;
    const long long ncells = (long long)nx * ny;
    const double* u = state + (long long)blockIdx.z * stride + (long long)var * ncells;
    const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
    double acc = 0.0;
    if (c < ncells && dims == 1) {
        const double uc = u[c];
        acc = add_power<P>(acc, uc - u[bc_value_index((int)c - h, nx, bc)], p);
        acc = add_power<P>(acc, uc - u[bc_value_index((int)c + h, nx, bc)], p);
    } else if (c < ncells) {
        const double uc = u[c];
        const int i = (int)(c % nx), j = (int)(c / nx);
        const bool wrap = bc == AVH_BC_PERIODIC;
        // count terms from cell k of a line of n on, s apart from one to the next
        auto line = [&](const double* v, int k, int n, long long s, int count) {
            int at = bc_value_index(k, n, bc);
            for (int t = 0; t < count; ++t) {
                acc = add_power<P>(acc, uc - v[at * s], p);
                ++k;
                if (wrap) at = at + 1 == n ? 0 : at + 1;
                else at = k < 0 ? 0 : (k > n - 1 ? n - 1 : k);
            }
        };
        for (int side = 0; side < (wrap ? 1 : 2); ++side) {
            line(u + bc_value_index(side ? i - h : i + h, nx, bc), j - h + 1, ny, nx, 2 * h - 1);
            line(u + (long long)bc_value_index(side ? j - h : j + h, ny, bc) * nx, i - h, nx, 1, 2 * h + 1);
        }
    }
    const double sum = block_sum(acc);
    if (threadIdx.x == 0)
        partial[((long long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = sum;
}

// Transposed copy of one variable of each sample: out[s][x][y] = u[s][y][x],
// 32 x 32 cells a workgroup through LDS.
__global__ __launch_bounds__(256) void transpose_kernel(const double* state, long long stride, int var, int nx, int ny,
                                                        double* out) {
    __shared__ double tile[32][33];
    const long long ncells = (long long)nx * ny;
    const double* u = state + (long long)blockIdx.z * stride + (long long)var * ncells;
    double* o = out + (long long)blockIdx.z * ncells;
    const int ntx = (nx + 31) / 32;
    const int x0 = ((int)blockIdx.x % ntx) * 32, y0 = ((int)blockIdx.x / ntx) * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8)
        if (x0 + tx < nx && y0 + r < ny) tile[r][tx] = u[(long long)(y0 + r) * nx + x0 + tx];
    __syncthreads();
    for (int r = ty; r < 32; r += 8)
        if (x0 + r < nx && y0 + tx < ny) o[(long long)(x0 + r) * ny + y0 + tx] = tile[tx][r];
}

// 2D.  The ring of lag h is two columns x -/+ h (y - h + 1 .. y + h - 1) and
// two rows y -/+ h (x - h .. x + h); a row of the field is a column of its
// transpose, so both are sweeps down a column: a lane owns a cell column and
// SWEEP_ROWS cells of it in registers, and every value loaded from column
// x + h serves all of them.  With periodic boundaries the pair at -h is the
// pair at +h seen from its other cell, so one side is swept and the finish
// doubles it; with neumann boundaries both are.
// Bound by the FP64 pipe (a subtraction and an FMA a pair for p = 2); the
// loads, one per SWEEP_ROWS pairs, come from L1 and L2.  16 samples of 256^2
// and 62 lags, periodic: 0.70 ms (60 % of the pipe), the gather of both sides
// 17.2 ms.
// Block = 64 columns x 4 * SWEEP_ROWS rows of one sample at one lag, of the
// field (blockIdx.x < cu) or of its transpose; the longest lags start first.
constexpr int SWEEP_ROWS = 8;

struct SweepParams {
    const double* state;  // sample 0's state; stride doubles from one sample to the next
    const double* trans;  // transposed copies
    long long stride;
    int var, nx, ny, bc;
    int cu;               // blocks covering the field, the others cover the transpose
    int nlags;            // lags 1 .. nlags
    double p;
    double* partial;      // [sample][lag][block]
};

template <int P>
__global__ __launch_bounds__(256) void structure_sweep_kernel(SweepParams S) {
    constexpr int R = SWEEP_ROWS;
    const int h = S.nlags - (int)blockIdx.y;
    const long long ncells = (long long)S.nx * S.ny;
    const bool flip = (int)blockIdx.x >= S.cu;
    const double* v = flip ? S.trans + (long long)blockIdx.z * ncells
                           : S.state + (long long)blockIdx.z * S.stride + (long long)S.var * ncells;
    const int nc = flip ? S.ny : S.nx, nr = flip ? S.nx : S.ny;  // columns, rows
    const int L = flip ? h : h - 1;
    const int tile = flip ? (int)blockIdx.x - S.cu : (int)blockIdx.x;
    const int ntx = (nc + 63) / 64;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int x = (tile % ntx) * 64 + lane;
    const int xc = x < nc ? x : nc - 1;
    const int y0 = ((tile / ntx) * 4 + wave) * R;
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0;
    if (y0 < nr) {
        double c[R];
#pragma unroll
        for (int r = 0; r < R; ++r) c[r] = v[(long long)(y0 + r < nr ? y0 + r : nr - 1) * nc + xc];
        const bool wrap = S.bc == AVH_BC_PERIODIC;
        for (int side = 0; side < (wrap ? 1 : 2); ++side) {
            const int xo = bc_value_index(side ? xc - h : xc + h, nc, S.bc);
            // rows y0 - L + t for t = 0 .. 2L + R - 1; row t meets the cells
            // r with t - 2L <= r <= t
            int k = y0 - L;
            int row = bc_value_index(k, nr, S.bc);
            auto next = [&]() {
                const double val = v[(long long)row * nc + xo];
                ++k;
                if (wrap) row = row + 1 == nr ? 0 : row + 1;
                else row = k < 0 ? 0 : (k > nr - 1 ? nr - 1 : k);
                return val;
            };
            if (2 * L >= R - 1) {
#pragma unroll
                for (int t = 0; t < R - 1; ++t) {
                    const double val = next();
#pragma unroll
                    for (int r = 0; r <= t; ++r) acc[r] = add_power<P>(acc[r], c[r] - val, S.p);
                }
                int left = 2 * L + 2 - R;
                for (; left >= 8; left -= 8) {
                    double val[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) val[i] = next();
#pragma unroll
                    for (int i = 0; i < 8; ++i)
#pragma unroll
                        for (int r = 0; r < R; ++r) acc[r] = add_power<P>(acc[r], c[r] - val[i], S.p);
                }
                for (; left > 0; --left) {
                    const double val = next();
#pragma unroll
                    for (int r = 0; r < R; ++r) acc[r] = add_power<P>(acc[r], c[r] - val, S.p);
                }
#pragma unroll
                for (int t = 1; t < R; ++t) {
                    const double val = next();
#pragma unroll
                    for (int r = t; r < R; ++r) acc[r] = add_power<P>(acc[r], c[r] - val, S.p);
                }
            } else {
                for (int t = 0; t < 2 * L + R; ++t) {
                    const double val = next();
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (r >= t - 2 * L && r <= t) acc[r] = add_power<P>(acc[r], c[r] - val, S.p);
                }
            }
        }
    }
    double sum = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (y0 + r < nr) sum = sum + acc[r];
    sum = block_sum(x < nc ? sum : 0.0);
    if (threadIdx.x == 0)
        S.partial[((long long)blockIdx.z * S.nlags + (h - 1)) * gridDim.x + blockIdx.x] = sum;
}

// out[s][0] = 0, out[s][h] = scale * (sum of the n partials of (s, h)), one
// wavefront each
__global__ __launch_bounds__(256) void structure_finish_kernel(const double* partial, int n, int nh, int nsamples,
                                                               double ncells, double factor, double* out) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (t >= nsamples * nh) return;
    const int s = t / nh, h = t % nh;
    double acc = 0.0;
    if (h > 0) {
        const double* q = partial + ((long long)s * (nh - 1) + (h - 1)) * n;
        for (int k = lane; k < n; k += 64) acc = acc + q[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc = acc + __shfl_xor(acc, off, 64);
    }
    if (lane == 0) out[t] = h > 0 ? factor * acc / ncells : 0.0;
}

// End time of every sample: samples with t < t_end (and no constraint
// failure) run again.
__global__ __launch_bounds__(256) void set_end_time_kernel(Control* ctrl, int nsamples, double t_end, int* active_count) {
    __shared__ int cnt;
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    for (int s = threadIdx.x; s < nsamples; s += 256) {
        Control* c = ctrl + s;
        c->t_end = t_end;
        c->active = (!(c->t >= t_end) && !c->violated) ? 1 : 0;
        if (c->active) atomicAdd(&cnt, 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) *active_count = cnt;
}

}  // namespace avh

namespace {

struct GroupHost {
    int n[3];
    int nsamples;
    long long ncells;
    double *A = nullptr, *B = nullptr, *C = nullptr;
    Control* ctrl = nullptr;
    double *mean_c = nullptr, *m2_c = nullptr, *mean_p = nullptr, *m2_p = nullptr;
    int* list = nullptr;
    int* list_len = nullptr;
    long long* counts = nullptr;
    int* active_count = nullptr;
};

template <class EQ>
void launch_batch_ew(const BatchParams& B, unsigned int nblocks, hipStream_t st) {
    hipLaunchKernelGGL(batch_ew_kernel<EQ>, dim3(nblocks), dim3(256), 0, st, B);
}
template <class EQ>
void launch_batch_stats(const StatsParams& S, unsigned int nblocks, hipStream_t st) {
    hipLaunchKernelGGL(batch_stats_kernel<EQ>, dim3(nblocks), dim3(256), 0, st, S);
}
typedef void (*BatchEw)(const BatchParams&, unsigned int, hipStream_t);
typedef void (*BatchStats)(const StatsParams&, unsigned int, hipStream_t);

BatchEw batch_ew_for(int eq) {
    switch (eq) {
    case AVH_EQ_BURGERS: return &launch_batch_ew<BurgersEq>;
    case AVH_EQ_EULER1: return &launch_batch_ew<EulerEq<1>>;
    case AVH_EQ_EULER2: return &launch_batch_ew<EulerEq<2>>;
    case AVH_EQ_EULER3: return &launch_batch_ew<EulerEq<3>>;
    }
    return nullptr;
}
BatchStats batch_stats_for(int eq) {
    switch (eq) {
    case AVH_EQ_BURGERS: return &launch_batch_stats<BurgersEq>;
    case AVH_EQ_EULER1: return &launch_batch_stats<EulerEq<1>>;
    case AVH_EQ_EULER2: return &launch_batch_stats<EulerEq<2>>;
    case AVH_EQ_EULER3: return &launch_batch_stats<EulerEq<3>>;
    }
    return nullptr;
}

}  // namespace

struct avh_batch {
    int device = 0;
    PinnedSlot slot;
    avh_config cfg{};
    int dim = 1, nv = 0;
    int ngroups = 0;
    GroupHost g[MAX_GROUPS];
    int nsaves = 0;         // statistics saves allocated
    int stats_adj = -1;     // adjuster index recording statistics
    int stats_initial = 0;  // record the initial state as save 0
    int initial_done = 0;
    Control proto{};        // per-sample initial Control
    hipStream_t stream = nullptr;
    BatchLauncher stage = nullptr;
    BatchEw ew = nullptr;
    BatchStats stats = nullptr;
    int graph_steps = 8;  // steps per captured hipGraph (0: ordinary launches)
    StepGraph graph;
    int shape = -1;       // tile shape of the stage kernel; -1: autotune on first use
    // groups the stage and element-wise launches cover: a group whose
    // samples have all stopped is dropped until the next avh_batch_advance
    bool live[MAX_GROUPS] = {true, true, true, true};
    // running samples per group, written by the end of a step into pinned
    // memory, and the marks after which avh_batch_advance reads them
    int* running = nullptr;
    hipEvent_t passed[2] = {nullptr, nullptr};
    // workspace of the observables (at most OBS_SLAB_BYTES and one sample's
    // share), kept until the batch goes; `obs_lock` serialises its users
    std::mutex obs_lock;
    double* work = nullptr;
    size_t work_cap = 0;
};

namespace {

void free_batch(avh_batch* b) {
    if (!b) return;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    b->graph.reset();
    for (int i = 0; i < b->ngroups; ++i) {
        GroupHost& G = b->g[i];
        (void)hipFree(G.A);
        (void)hipFree(G.B);
        (void)hipFree(G.C);
        (void)hipFree(G.ctrl);
        (void)hipFree(G.mean_c);
        (void)hipFree(G.m2_c);
        (void)hipFree(G.mean_p);
        (void)hipFree(G.m2_p);
        (void)hipFree(G.list);
        (void)hipFree(G.list_len);
        (void)hipFree(G.counts);
        (void)hipFree(G.active_count);
    }
    (void)hipFree(b->work);
    for (hipEvent_t e : b->passed)
        if (e) (void)hipEventDestroy(e);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

// Samples of an observable are taken in slabs whose workspace stays below this
// (or one sample at a time where a sample needs more).
constexpr size_t OBS_SLAB_BYTES = (size_t)64 << 20;

int slab_samples(size_t doubles_per_sample, int nsamples) {
    const size_t per = doubles_per_sample * sizeof(double);
    const size_t fit = per ? OBS_SLAB_BYTES / per : (size_t)nsamples;
    return (int)std::max<size_t>(1, std::min<size_t>(fit, (size_t)nsamples));
}

// b->work with room for n doubles (b->obs_lock is held)
avh_status ensure_work(avh_batch* b, size_t n) {
    if (n <= b->work_cap) return AVH_OK;
    (void)hipFree(b->work);
    b->work = nullptr;
    b->work_cap = 0;
    if (hipMalloc(&b->work, sizeof(double) * n) != hipSuccess) {
        b->work = nullptr;
        (void)hipGetLastError();
        return fail(AVH_ENOMEM, "device allocation failed");
    }
    b->work_cap = n;
    return AVH_OK;
}

// Launch parameters over the live groups (slot j of P is group index[j]);
// nblocks = the launch's block count (8 * per_xcd for a stage launch, the
// element-wise blocks of every sample otherwise), 0 if no group is live.
BatchParams batch_params(const avh_batch* b, int mode, bool ew_blocks, unsigned int* nblocks,
                         int* index = nullptr) {
    BatchParams P;
    std::memset(&P, 0, sizeof P);
    P.bc = b->cfg.boundary;
    P.mode = mode;
    P.gamma = b->cfg.gamma;
    unsigned int first = 0;
    unsigned int per_xcd[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int j = 0;
    for (int i = 0; i < b->ngroups; ++i) {
        if (!b->live[i]) continue;
        const GroupHost& G = b->g[i];
        GroupDesc& D = P.g[j];
        if (index) index[j] = i;
        ++j;
        D.ctrl = G.ctrl;
        D.stride = (long long)b->nv * G.ncells;
        D.ncells = G.ncells;
        for (int d = 0; d < 3; ++d) D.n[d] = G.n[d];
        D.tiles = ew_blocks ? (unsigned int)((G.ncells + 255) / 256) : stage_tiles(G.n, b->dim, b->shape);
        D.first_block = first;
        D.nsamples = G.nsamples;
        first += D.tiles * (unsigned int)G.nsamples;
        for (unsigned int x = 0; x < 8; ++x) per_xcd[x] += xcd_samples(G.nsamples, x) * D.tiles;
    }
    P.ngroups = j;
    P.per_xcd = 0;
    for (unsigned int x = 0; x < 8; ++x) P.per_xcd = std::max(P.per_xcd, per_xcd[x]);
    *nblocks = ew_blocks ? first : 8u * P.per_xcd;
    return P;
}

StatsParams stats_params(const avh_batch* b, unsigned int* nblocks) {
    StatsParams S;
    std::memset(&S, 0, sizeof S);
    S.ngroups = b->ngroups;
    S.stats_adj = b->stats_adj;
    S.save_offset = b->stats_initial ? 0 : 1;
    S.gamma = b->cfg.gamma;
    unsigned int first = 0;
    for (int i = 0; i < b->ngroups; ++i) {
        const GroupHost& G = b->g[i];
        StatsGroup& T = S.g[i];
        T.ctrl = G.ctrl;
        T.state = G.A;
        T.stride = (long long)b->nv * G.ncells;
        T.ncells = G.ncells;
        T.nsamples = G.nsamples;
        T.nsaves = b->nsaves;
        T.list = G.list;
        T.list_len = G.list_len;
        T.counts = G.counts;
        T.active_count = G.active_count;
        T.host_active = b->running + i;
        T.mean_c = G.mean_c;
        T.m2_c = G.m2_c;
        T.mean_p = G.mean_p;
        T.m2_p = G.m2_p;
        T.blocks = (unsigned int)((G.ncells + 255) / 256);
        T.first_block = first;
        first += T.blocks;
    }
    *nblocks = first;
    return S;
}

TuneKey batch_key(const avh_batch* b) {
    long long total = 0;
    for (int i = 0; i < b->ngroups; ++i) total += b->g[i].nsamples;
    return tune_key(TUNE_BATCH, b->cfg, b->dim, {b->g[0].n[0], b->g[0].n[1], total});
}

// Times every tile shape over all samples with the first stage (flux-only if
// every sample has stopped) and, for RK2 and RK3, the second stage, and keeps the
// fastest.  They write the L0 and U2 buffers and add to the per-sample
// wave-speed maxima; the control blocks are restored afterwards.
void set_all_live(avh_batch* b);

avh_status batch_autotune(avh_batch* b, int* best, double* ms, int* nshapes) {
    const int ns = num_shapes(b->dim);
    set_all_live(b);  // time the launches over every group
    AVH_HIP(hipStreamSynchronize(b->stream));
    std::vector<std::vector<Control>> saved(b->ngroups);
    for (int i = 0; i < b->ngroups; ++i) {
        saved[i].resize(b->g[i].nsamples);
        AVH_HIP(hipMemcpy(saved[i].data(), b->g[i].ctrl, sizeof(Control) * b->g[i].nsamples,
                          hipMemcpyDeviceToHost));
    }
    bool active = false;
    for (const auto& cs : saved)
        for (const Control& c : cs) active = active || c.active;
    const bool second = active && b->cfg.integrator != AVH_INT_FORWARDEULER;
    const int keep = b->shape;
    int bst = 0;
    double tmin = 0;
    avh_status r = AVH_OK;
    for (int k = 0; k < ns && r == AVH_OK; ++k) {
        double t = 0;
        if (ns > 1) {
            b->shape = k;
            unsigned int nb = 0;
            BatchParams P = batch_params(b, active ? MODE_L : MODE_FLUX_ONLY, false, &nb);
            BatchParams P2 =
                batch_params(b, b->cfg.integrator == AVH_INT_RUNGEKUTTA3 ? MODE_RK3_2 : MODE_RK2_2, false, &nb);
            for (int i = 0; i < b->ngroups; ++i) {
                P.g[i].in = P.g[i].u0 = P2.g[i].u0 = b->g[i].A;
                P.g[i].out = b->g[i].B;
                if (b->cfg.integrator == AVH_INT_RUNGEKUTTA2) P.g[i].copy = b->g[i].C;
                P2.g[i].in = b->g[i].B;
                P2.g[i].out = b->g[i].C;
            }
            r = time_launches(b->stream, 3,
                              [&]() {
                                  hipError_t e = b->stage(P, nb, k, b->stream);
                                  if (e == hipSuccess && second) e = b->stage(P2, nb, k, b->stream);
                                  return e;
                              },
                              &t);
        }
        if (ms) ms[k] = t;
        if (k == 0 || t < tmin) {
            tmin = t;
            bst = k;
        }
    }
    b->shape = keep;
    AVH_HIP(hipStreamSynchronize(b->stream));
    for (int i = 0; i < b->ngroups; ++i)
        AVH_HIP(hipMemcpy(b->g[i].ctrl, saved[i].data(), sizeof(Control) * b->g[i].nsamples,
                          hipMemcpyHostToDevice));
    if (r) return r;
    if (b->shape != bst) b->graph.reset();
    b->shape = bst;
    tune_store(batch_key(b), bst, active);
    if (best) *best = bst;
    if (nshapes) *nshapes = ns;
    return AVH_OK;
}

avh_status batch_ensure_shape(avh_batch* b) {
    if (b->shape >= 0) return AVH_OK;
    int s;
    if (tune_lookup(batch_key(b), &s)) {
        b->shape = s;
        return AVH_OK;
    }
    return batch_autotune(b, nullptr, nullptr, nullptr);
}

// Launches per batch step: the stages (plus forward euler's element-wise
// pass), the end-of-step kernel and, with statistics, the statistics kernel.
int batch_launches_per_step(const avh_batch* b) {
    const int stages = b->cfg.integrator == AVH_INT_RUNGEKUTTA3 ? 3 : 2;
    return stages + 1 + (b->nsaves > 0 ? 1 : 0);
}

void set_all_live(avh_batch* b) {
    bool changed = false;
    for (int i = 0; i < b->ngroups; ++i) {
        changed = changed || !b->live[i];
        b->live[i] = true;
    }
    if (changed) b->graph.reset();
}

avh_status enqueue_batch_step(avh_batch* b, EventMarks* tm = nullptr) {
    avh_status r;
    if ((r = mark(tm, b->stream))) return r;
    unsigned int nb = 0, nbe = 0;
    int index[MAX_GROUPS] = {0, 0, 0, 0};
    auto set_ptrs = [&](BatchParams& P, int which_in, int which_u0, int which_out) {
        for (int j = 0; j < P.ngroups; ++j) {
            const GroupHost& G = b->g[index[j]];
            double* bufs[3] = {G.A, G.B, G.C};
            P.g[j].in = bufs[which_in];
            P.g[j].u0 = bufs[which_u0];
            P.g[j].out = bufs[which_out];
        }
    };
    // a launch with no live group is left out (every sample has stopped;
    // the end-of-step kernel then leaves them unchanged)
    auto stage = [&](BatchParams& P) -> avh_status {
        if (nb) AVH_HIP(b->stage(P, nb, b->shape, b->stream));
        return mark(tm, b->stream);
    };
    enum { A = 0, B = 1, C = 2 };
    BatchParams P = batch_params(b, MODE_L, false, &nb, index);
    set_ptrs(P, A, A, B);
    if (b->cfg.integrator == AVH_INT_RUNGEKUTTA2)
        for (int j = 0; j < P.ngroups; ++j) P.g[j].copy = b->g[index[j]].C;
    if ((r = stage(P))) return r;
    if (b->cfg.integrator == AVH_INT_FORWARDEULER) {
        BatchParams E = batch_params(b, MODE_L, true, &nbe, index);
        set_ptrs(E, B, A, A);
        if (nbe) {
            b->ew(E, nbe, b->stream);
            AVH_HIP(hipGetLastError());
        }
        if ((r = mark(tm, b->stream))) return r;
    } else if (b->cfg.integrator == AVH_INT_RUNGEKUTTA2) {
        P = batch_params(b, MODE_RK2_2, false, &nb, index);
        set_ptrs(P, B, C, A);
        if ((r = stage(P))) return r;
    } else {
        P = batch_params(b, MODE_RK3_2, false, &nb, index);
        set_ptrs(P, B, A, C);
        if ((r = stage(P))) return r;
        P = batch_params(b, MODE_RK3_3, false, &nb, index);
        set_ptrs(P, C, A, A);
        if ((r = stage(P))) return r;
    }
    unsigned int nbs = 0;
    StatsParams S = stats_params(b, &nbs);
    int maxs = 64;
    for (int i = 0; i < b->ngroups; ++i) maxs = std::max(maxs, std::min(1024, (b->g[i].nsamples + 63) / 64 * 64));
    hipLaunchKernelGGL(batch_finish_kernel, dim3(b->ngroups), dim3(maxs), 0, b->stream, S);
    AVH_HIP(hipGetLastError());
    if ((r = mark(tm, b->stream))) return r;
    if (b->nsaves > 0) {
        b->stats(S, nbs, b->stream);
        AVH_HIP(hipGetLastError());
        if ((r = mark(tm, b->stream))) return r;
    }
    return AVH_OK;
}

}  // namespace

extern "C" {

avh_status avh_batch_create(avh_ctx* ctx, const avh_config* cfg, int ngroups, const avh_group* groups,
                            double t_end, int stats_saves, int stats_write_initial, avh_batch** out) {
    if (!ctx || !cfg || !groups || !out) return fail(AVH_EINVAL, "null argument");
    *out = nullptr;
    if (ngroups < 1 || ngroups > MAX_GROUPS) return fail(AVH_EINVAL, "1 to 4 resolution groups");
    const int nv = nvars_of(cfg->equation);
    const int ng = ghosts_of(cfg->reconstruction);
    if (!nv || !ng) return fail(AVH_EINVAL, "unknown equation or reconstruction");
    if (cfg->integrator < AVH_INT_FORWARDEULER || cfg->integrator > AVH_INT_RUNGEKUTTA3)
        return fail(AVH_EINVAL, "unknown integrator");
    if (cfg->boundary != AVH_BC_PERIODIC && cfg->boundary != AVH_BC_NEUMANN)
        return fail(AVH_EINVAL, "unknown boundary");
    if (stats_saves < 0) return fail(AVH_EINVAL, "stats_saves must be >= 0");
    int dim = 0;
    for (int i = 0; i < ngroups; ++i) {
        const avh_group& G = groups[i];
        if (G.nsamples < 1) return fail(AVH_EINVAL, "every group needs at least one sample");
        for (int d = 0; d < 3; ++d)
            if (G.n[d] < 1) return fail(AVH_EINVAL, "grid sizes must be >= 1");
        const int gd = G.n[2] > 1 ? 3 : (G.n[1] > 1 ? 2 : 1);
        if (dim && gd != dim) return fail(AVH_EINVAL, "all groups need the same number of active axes");
        dim = gd;
        for (int d = 0; d < dim; ++d)
            if (G.n[d] < ng) return fail(AVH_EINVAL, "too few cells for the ghost width");
    }
    const Launchers L = launchers_for(cfg->equation, cfg->reconstruction, cfg->flux, dim);
    if (!L.batch)
        return fail(AVH_EINVAL,
                    "unsupported combination for batched runs (1D or 2D grids; burgers: godunov; euler<n>: hll, hll3)");
    AVH_HIP(hipSetDevice(ctx->device));
    auto b = new (std::nothrow) avh_batch;
    if (!b) return fail(AVH_ENOMEM, "host allocation failed");
    b->device = ctx->device;
    b->cfg = *cfg;
    b->dim = dim;
    b->nv = nv;
    b->ngroups = ngroups;
    b->stage = L.batch;
    b->ew = batch_ew_for(cfg->equation);
    b->stats = batch_stats_for(cfg->equation);
    b->stats_initial = stats_write_initial ? 1 : 0;
    b->nsaves = stats_saves > 0 ? stats_saves + b->stats_initial : 0;
    Control& h = b->proto;
    std::memset(&h, 0, sizeof h);
    h.cfl = cfg->cfl;
    h.t_end = t_end;
    if (stats_saves > 0) {
        // FixedIntervalStatistics: interval endTime/numberOfSaves, no start
        // offset (alsuq/src/config/Setup.cpp:270-285,
        // alsuq/src/stats/FixedIntervalStatistics.cpp:33-41)
        b->stats_adj = 0;
        h.n_adj = 1;
        h.adj_interval[0] = t_end / stats_saves;
        h.adj_start[0] = 0;
        h.adj_saved[0] = stats_write_initial ? 0 : 1;
    }
    h.active = (0.0 < t_end) ? 1 : 0;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
        b->stream = nullptr;
        free_batch(b);
        return fail(AVH_EHIP, "hipStreamCreate failed");
    }
    bool marks = (b->running = (int*)b->slot.take(ctx->pinned)) != nullptr;
    for (hipEvent_t& e : b->passed) marks = marks && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!marks) {
        free_batch(b);
        return fail(AVH_ENOMEM, "host allocation failed");
    }
    for (int i = 0; i < ngroups; ++i) {
        GroupHost& G = b->g[i];
        for (int d = 0; d < 3; ++d) G.n[d] = groups[i].n[d];
        G.nsamples = groups[i].nsamples;
        G.ncells = (long long)G.n[0] * G.n[1] * G.n[2];
        const size_t state = (size_t)nv * G.ncells * G.nsamples * sizeof(double);
        const size_t stat = (size_t)std::max(1, b->nsaves) * nv * G.ncells * sizeof(double);
        bool ok = hipMalloc(&G.A, state) == hipSuccess && hipMalloc(&G.B, state) == hipSuccess &&
                  hipMalloc(&G.C, state) == hipSuccess &&
                  hipMalloc(&G.ctrl, sizeof(Control) * G.nsamples) == hipSuccess &&
                  hipMalloc(&G.mean_c, stat) == hipSuccess && hipMalloc(&G.m2_c, stat) == hipSuccess &&
                  hipMalloc(&G.mean_p, stat) == hipSuccess && hipMalloc(&G.m2_p, stat) == hipSuccess &&
                  hipMalloc(&G.list, sizeof(int) * 3 * G.nsamples) == hipSuccess &&
                  hipMalloc(&G.list_len, sizeof(int)) == hipSuccess &&
                  hipMalloc(&G.counts, sizeof(long long) * std::max(1, b->nsaves)) == hipSuccess &&
                  hipMalloc(&G.active_count, sizeof(int)) == hipSuccess;
        if (!ok) {
            b->ngroups = i + 1;
            free_batch(b);
            return fail(AVH_ENOMEM, "device allocation failed");
        }
        ok = hipMemset(G.A, 0, state) == hipSuccess && hipMemset(G.B, 0, state) == hipSuccess &&
             hipMemset(G.C, 0, state) == hipSuccess && hipMemset(G.mean_c, 0, stat) == hipSuccess &&
             hipMemset(G.m2_c, 0, stat) == hipSuccess && hipMemset(G.mean_p, 0, stat) == hipSuccess &&
             hipMemset(G.m2_p, 0, stat) == hipSuccess && hipMemset(G.list_len, 0, sizeof(int)) == hipSuccess &&
             hipMemset(G.counts, 0, sizeof(long long) * std::max(1, b->nsaves)) == hipSuccess;
        Control c = h;
        for (int d = 0; d < 3; ++d) c.cell[d] = (cfg->upper[d] - cfg->lower[d]) / double(G.n[d]);
        if (G.n[1] == 1) c.cell[1] = 1;
        if (G.n[2] == 1) c.cell[2] = 1;
        std::vector<Control> cs(G.nsamples, c);
        const int act = c.active ? G.nsamples : 0;
        ok = ok && hipMemcpy(G.ctrl, cs.data(), sizeof(Control) * G.nsamples, hipMemcpyHostToDevice) == hipSuccess &&
             hipMemcpy(G.active_count, &act, sizeof(int), hipMemcpyHostToDevice) == hipSuccess;
        if (!ok) {
            b->ngroups = i + 1;
            free_batch(b);
            return fail(AVH_EHIP, "device initialisation failed");
        }
    }
    *out = b;
    return AVH_OK;
}

avh_status avh_batch_destroy(avh_batch* b) {
    free_batch(b);
    return AVH_OK;
}

avh_status avh_batch_add_fixed_interval_adjuster(avh_batch* b, double interval, double start, int write_initial) {
    if (!b) return fail(AVH_EINVAL, "null argument");
    if (!(interval > 0)) return fail(AVH_EINVAL, "interval must be positive");
    if (b->proto.n_adj >= MAX_ADJ) return fail(AVH_EINVAL, "at most 4 adjusters");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    const int i = b->proto.n_adj++;
    b->proto.adj_interval[i] = interval;
    b->proto.adj_start[i] = start;
    b->proto.adj_saved[i] = write_initial ? 0 : 1;
    // the Runner's callWriters() at t = 0 (alsuq/src/run/Runner.cpp:68)
    if (0.0 >= (double)b->proto.adj_saved[i] * interval + start) b->proto.adj_saved[i] += 1;
    for (int k = 0; k < b->ngroups; ++k) {
        GroupHost& G = b->g[k];
        std::vector<Control> cs(G.nsamples);
        AVH_HIP(hipMemcpy(cs.data(), G.ctrl, sizeof(Control) * G.nsamples, hipMemcpyDeviceToHost));
        for (auto& c : cs) {
            c.n_adj = b->proto.n_adj;
            c.adj_interval[i] = interval;
            c.adj_start[i] = start;
            c.adj_saved[i] = b->proto.adj_saved[i];
        }
        AVH_HIP(hipMemcpy(G.ctrl, cs.data(), sizeof(Control) * G.nsamples, hipMemcpyHostToDevice));
    }
    return AVH_OK;
}

static avh_status check_gs(const avh_batch* b, int group, int sample) {
    if (!b) return fail(AVH_EINVAL, "null argument");
    if (group < 0 || group >= b->ngroups) return fail(AVH_EINVAL, "no such group");
    if (sample < 0 || sample >= b->g[group].nsamples) return fail(AVH_EINVAL, "no such sample");
    return AVH_OK;
}

avh_status avh_batch_set_state(avh_batch* b, int group, int sample, const double* host_interior) {
    avh_status r = check_gs(b, group, sample);
    if (r) return r;
    if (!host_interior) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    const GroupHost& G = b->g[group];
    const size_t n = (size_t)b->nv * G.ncells;
    AVH_HIP(hipMemcpy(G.A + (size_t)sample * n, host_interior, n * sizeof(double), hipMemcpyHostToDevice));
    return AVH_OK;
}

avh_status avh_batch_get_state(avh_batch* b, int group, int sample, double* host_interior) {
    avh_status r = check_gs(b, group, sample);
    if (r) return r;
    if (!host_interior) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    const GroupHost& G = b->g[group];
    const size_t n = (size_t)b->nv * G.ncells;
    AVH_HIP(hipMemcpy(host_interior, G.A + (size_t)sample * n, n * sizeof(double), hipMemcpyDeviceToHost));
    return AVH_OK;
}

avh_status avh_batch_set_kh2d(avh_batch* b, int group, const double* host_interfaces) {
    avh_status r = check_gs(b, group, 0);
    if (r) return r;
    if (!host_interfaces) return fail(AVH_EINVAL, "null argument");
    if (b->cfg.equation != AVH_EQ_EULER2 || b->dim != 2) return fail(AVH_EINVAL, "KH fill needs euler2 on 2D grids");
    AVH_HIP(hipSetDevice(b->device));
    const GroupHost& G = b->g[group];
    const size_t bytes = (size_t)G.nsamples * 2 * G.n[0] * sizeof(double);
    double* d = nullptr;
    AVH_HIP(hipMalloc(&d, bytes));
    hipError_t e = hipMemcpy(d, host_interfaces, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        const double dy = (b->cfg.upper[1] - b->cfg.lower[1]) / double(G.n[1]);
        hipLaunchKernelGGL(kh2d_fill_kernel, dim3(2048), dim3(256), 0, b->stream, G.A, (long long)b->nv * G.ncells,
                           G.n[0], G.n[1], d, G.nsamples, b->cfg.lower[1], dy, b->cfg.gamma);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
    (void)hipFree(d);
    if (e != hipSuccess) return fail(AVH_EHIP, std::string("KH fill: ") + hipGetErrorString(e));
    return AVH_OK;
}

// Enqueues n steps.  They go out a graph's worth at a time, two ahead of the
// device, so that what would follow the last sample's end is not launched at
// all: a launch in which every sample has stopped still deals all its
// workgroups (84 samples of 128^2 to 512^2: 9 us, and three of them a step).
static avh_status enqueue_until_stopped(avh_batch* b, int64_t n) {
    const int64_t unit = b->graph_steps >= 2 ? b->graph_steps : 8;
    for (int64_t k = 0; n > 0; ++k, n -= unit) {
        const hipEvent_t mark = b->passed[k % 2];
        if (k >= 2) {
            AVH_HIP(hipEventSynchronize(mark));
            int running = 0;
            for (int i = 0; i < b->ngroups; ++i) running += __atomic_load_n(b->running + i, __ATOMIC_RELAXED);
            if (running == 0) return AVH_OK;
        }
        const avh_status r = enqueue_steps_graphed(b->graph, b->graph_steps, b->stream, std::min<int64_t>(n, unit),
                                                   [b]() { return enqueue_batch_step(b); });
        if (r) return r;
        AVH_HIP(hipEventRecord(mark, b->stream));
    }
    return AVH_OK;
}

avh_status avh_batch_advance(avh_batch* b, int64_t max_steps, int chunk, int64_t* steps_done, int64_t* active_left) {
    if (!b) return fail(AVH_EINVAL, "null argument");
    if (chunk < 1) chunk = 1;
    AVH_HIP(hipSetDevice(b->device));
    if (b->stats_initial && !b->initial_done && b->nsaves > 0) {
        unsigned int nbs = 0;
        StatsParams S = stats_params(b, &nbs);
        hipLaunchKernelGGL(batch_initial_save_kernel, dim3(b->ngroups), dim3(256), 0, b->stream, S);
        AVH_HIP(hipGetLastError());
        b->stats(S, nbs, b->stream);
        AVH_HIP(hipGetLastError());
        b->initial_done = 1;
    }
    avh_status rs = batch_ensure_shape(b);
    if (rs) return rs;
    // every group takes part until a chunk shows that all its samples have
    // stopped (the end-of-step kernel counts the running samples of every
    // group, live or not, at every step)
    set_all_live(b);
    int64_t done = 0, left = 0;
    while (done < max_steps) {
        const int64_t k = std::min<int64_t>(chunk, max_steps - done);
        const avh_status r = enqueue_until_stopped(b, k);
        if (r) return r;
        done += k;
        AVH_HIP(hipStreamSynchronize(b->stream));
        left = 0;
        for (int i = 0; i < b->ngroups; ++i) {
            int a = 0;
            AVH_HIP(hipMemcpy(&a, b->g[i].active_count, sizeof(int), hipMemcpyDeviceToHost));
            left += a;
            if (a == 0 && b->live[i]) {
                b->live[i] = false;  // drop the finished group from the launches
                b->graph.reset();
            }
        }
        if (left == 0) break;
    }
    if (steps_done) *steps_done = done;
    if (active_left) *active_left = left;
    return AVH_OK;
}

avh_status avh_batch_set_graph_steps(avh_batch* b, int steps) {
    if (!b || steps < 0 || steps > 4096) return fail(AVH_EINVAL, "bad argument");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    b->graph.reset();
    b->graph_steps = steps;
    return AVH_OK;
}

avh_status avh_batch_violations(avh_batch* b, int group, int64_t* count, int64_t* first_sample) {
    avh_status r = check_gs(b, group, 0);
    if (r) return r;
    if (!count || !first_sample) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    const GroupHost& G = b->g[group];
    std::vector<Control> cs(G.nsamples);
    AVH_HIP(hipMemcpy(cs.data(), G.ctrl, sizeof(Control) * G.nsamples, hipMemcpyDeviceToHost));
    *count = 0;
    *first_sample = -1;
    for (int s = 0; s < G.nsamples; ++s)
        if (cs[s].violated) {
            if (*first_sample < 0) *first_sample = s;
            *count += 1;
        }
    return AVH_OK;
}

avh_status avh_batch_set_end_time(avh_batch* b, double t_end) {
    if (!b) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(b->device));
    for (int i = 0; i < b->ngroups; ++i) {
        hipLaunchKernelGGL(set_end_time_kernel, dim3(1), dim3(256), 0, b->stream, b->g[i].ctrl, b->g[i].nsamples, t_end,
                           b->g[i].active_count);
        AVH_HIP(hipGetLastError());
    }
    b->proto.t_end = t_end;
    AVH_HIP(hipStreamSynchronize(b->stream));
    return AVH_OK;
}

avh_status avh_batch_kinetic_energy(avh_batch* b, int group, int component, double* out) {
    avh_status r = check_gs(b, group, 0);
    if (r) return r;
    if (!out) return fail(AVH_EINVAL, "null argument");
    if (b->cfg.equation == AVH_EQ_BURGERS || component < 0 || component >= b->nv - 2)
        return fail(AVH_EINVAL, "kinetic energy needs an euler equation and a velocity component < dimensions");
    AVH_HIP(hipSetDevice(b->device));
    const GroupHost& G = b->g[group];
    double dv = 1.0;
    for (int d = 0; d < 3; ++d)
        if (G.n[d] > 1) dv *= (b->cfg.upper[d] - b->cfg.lower[d]) / double(G.n[d]);
    std::lock_guard<std::mutex> lock(b->obs_lock);
    // 2048 cells a block: 8 a thread
    const int nblk = (int)std::max<long long>(1, std::min<long long>((G.ncells + 2047) / 2048, 1024));
    const int slab = std::min(slab_samples((size_t)nblk + 1, G.nsamples), 65535);
    if ((r = ensure_work(b, (size_t)slab * (nblk + 1)))) return r;
    double* d = b->work + (size_t)slab * nblk;
    const long long stride = (long long)b->nv * G.ncells;
    for (int s0 = 0; s0 < G.nsamples; s0 += slab) {
        const int m = std::min(slab, G.nsamples - s0);
        hipLaunchKernelGGL(kinetic_energy_kernel, dim3(nblk, m), dim3(256), 0, b->stream, G.A + s0 * stride, stride,
                           G.ncells, component, dv, nblk == 1 ? d : b->work);
        AVH_HIP(hipGetLastError());
        if (nblk > 1) {
            hipLaunchKernelGGL(sums_finish_kernel, dim3((m + 3) / 4), dim3(256), 0, b->stream, b->work, nblk, m, dv, d);
            AVH_HIP(hipGetLastError());
        }
        AVH_HIP(hipMemcpyAsync(out + s0, d, sizeof(double) * m, hipMemcpyDeviceToHost, b->stream));
        AVH_HIP(hipStreamSynchronize(b->stream));
    }
    return AVH_OK;
}

// blocks of a sweep of columns of nr cells, nc of them, and of its transpose
static int sweep_blocks(int nc, int nr) { return ((nc + 63) / 64) * ((nr + 4 * SWEEP_ROWS - 1) / (4 * SWEEP_ROWS)); }

// Whether a 2D structure function sweeps columns, or gathers a cell a thread.
// The sweep saves loads and indices; it takes a transposed copy first, and
// lanes and rows past the grid's edge are lost.  us of a call, gather / sweep:
//   p = 2     1 lag     256^2 x 16 32 / 40, 1000x800 40 / 41, 17x300 x 3 26 / 31
//             6 lags    256^2 x 16 82 / 62, 128^2 x 4 30 / 33, 17x300 x 3 29 / 33
//             16 lags   128^2 x 4 46 / 36, 17x300 x 3 34 / 35, 16^2 31 / 32
//             32 lags   256^2 x 16 975 / 247, 17x300 x 3 48 / 42, 16^2 36 / 34
// so the gather takes calls of few lags and few pairs of cells.
//   p = 2.5 is bound by the powers, whichever way the cells come: neumann
//             62 lags   17x300 x 3 1565 / 3975, 130^2 x 8 11306 / 16474,
//                       256^2 10760 (2 samples) / 9497
//             8 lags    256^2 x 2 237 / 291, x 16 1645 / 1551, 1000x800 1296 / 1211
//   and p = 1.5, periodic
//             3 lags    256^2 x 16 181 / 197, x 64 621 / 607, 512^2 x 8 325 / 318
//             6 lags    256^2 x 8 274 / 289, x 16 517 / 505, x 64 1975 / 1807
//             8 lags    128^2 x 64 868 / 955, 256^2 x 2 135 / 161, x 8 442 / 442
// so there the sweep takes only grids that fill its lanes, in enough blocks: more
// of them where the lags are few.
static bool structure_sweeps(bool general, int nx, int ny, int nsamples, int nlags) {
    const long long cells = (long long)nx * ny;
    if (!general) return nlags > 12 || cells * nsamples * (4 * nlags * (nlags + 1)) > (1ll << 24);
    const int cu = sweep_blocks(nx, ny), ct = sweep_blocks(ny, nx);
    const double slots = 64.0 * 4 * SWEEP_ROWS * (cu + ct);  // lanes times rows of the field's sweep and the transpose's
    const long long blocks = (long long)(cu + ct) * nlags * nsamples;
    const int n = std::min(nx, ny);
    return 2 * cells >= 0.92 * slots &&
           ((nlags >= 8 && n >= 128 && blocks >= 2048) || (nlags >= 3 && n > 128 && blocks >= 6144));
}

static avh_status launch_structure_gather(int pi, dim3 grid, hipStream_t st, const double* state, long long stride,
                                        int var, int nx, int ny, int dims, int bc, double p, double* partial) {
    switch (pi) {
    case 1: hipLaunchKernelGGL(structure_gather_kernel<1>, grid, dim3(256), 0, st, state, stride, var, nx, ny, dims, bc, p, partial); break;
    case 2: hipLaunchKernelGGL(structure_gather_kernel<2>, grid, dim3(256), 0, st, state, stride, var, nx, ny, dims, bc, p, partial); break;
    case 3: hipLaunchKernelGGL(structure_gather_kernel<3>, grid, dim3(256), 0, st, state, stride, var, nx, ny, dims, bc, p, partial); break;
    case 4: hipLaunchKernelGGL(structure_gather_kernel<4>, grid, dim3(256), 0, st, state, stride, var, nx, ny, dims, bc, p, partial); break;
    case 5: hipLaunchKernelGGL(structure_gather_kernel<5>, grid, dim3(256), 0, st, state, stride, var, nx, ny, dims, bc, p, partial); break;
    default: hipLaunchKernelGGL(structure_gather_kernel<0>, grid, dim3(256), 0, st, state, stride, var, nx, ny, dims, bc, p, partial); break;
    }
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

static avh_status launch_structure_sweep(int pi, dim3 grid, hipStream_t st, const SweepParams& S) {
    switch (pi) {
    case 1: hipLaunchKernelGGL(structure_sweep_kernel<1>, grid, dim3(256), 0, st, S); break;
    case 2: hipLaunchKernelGGL(structure_sweep_kernel<2>, grid, dim3(256), 0, st, S); break;
    case 3: hipLaunchKernelGGL(structure_sweep_kernel<3>, grid, dim3(256), 0, st, S); break;
    case 4: hipLaunchKernelGGL(structure_sweep_kernel<4>, grid, dim3(256), 0, st, S); break;
    case 5: hipLaunchKernelGGL(structure_sweep_kernel<5>, grid, dim3(256), 0, st, S); break;
    default: hipLaunchKernelGGL(structure_sweep_kernel<0>, grid, dim3(256), 0, st, S); break;
    }
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

avh_status avh_batch_structure_cube(avh_batch* b, int group, int var, int number_of_h, double p, double* out) {
    avh_status r = check_gs(b, group, 0);
    if (r) return r;
    if (!out) return fail(AVH_EINVAL, "null argument");
    if (var < 0 || var >= b->nv) return fail(AVH_EINVAL, "no such variable");
    if (b->dim > 2) return fail(AVH_EINVAL, "structure functions of batches: 1D and 2D grids");
    const GroupHost& G = b->g[group];
    if (number_of_h < 2 || number_of_h > 65535) return fail(AVH_EINVAL, "number_of_h must be in [2, 65535]");
    if (!(p > 0)) return fail(AVH_EINVAL, "p must be positive");
    if (G.nsamples > 65535) return fail(AVH_EINVAL, "structure functions: at most 65535 samples per group");
    AVH_HIP(hipSetDevice(b->device));
    const int nx = G.n[0], ny = G.n[1], nlags = number_of_h - 1;
    const int pi = p == 1.0 ? 1 : p == 2.0 ? 2 : p == 3.0 ? 3 : p == 4.0 ? 4 : p == 5.0 ? 5 : 0;
    const bool two = b->dim == 2 && structure_sweeps(pi == 0, nx, ny, G.nsamples, nlags);
    const int cu = two ? sweep_blocks(nx, ny) : (int)((G.ncells + 255) / 256);
    const int ct = two ? sweep_blocks(ny, nx) : 0;
    const size_t npart = (size_t)(cu + ct) * nlags;
    const size_t per = npart + (two ? (size_t)G.ncells : 0) + number_of_h;
    const int slab = slab_samples(per, G.nsamples);
    std::lock_guard<std::mutex> lock(b->obs_lock);
    if ((r = ensure_work(b, per * slab))) return r;
    double* const part = b->work;
    double* const trans = part + npart * slab;
    double* const d = trans + (two ? (size_t)G.ncells * slab : 0);
    const long long stride = (long long)b->nv * G.ncells;
    for (int s0 = 0; s0 < G.nsamples; s0 += slab) {
        const int m = std::min(slab, G.nsamples - s0);
        const double* state = G.A + s0 * stride;
        if (two) {
            hipLaunchKernelGGL(transpose_kernel, dim3(((nx + 31) / 32) * ((ny + 31) / 32), 1, m), dim3(256), 0, b->stream,
                               state, stride, var, nx, ny, trans);
            AVH_HIP(hipGetLastError());
            SweepParams S;
            S.state = state;
            S.trans = trans;
            S.stride = stride;
            S.var = var;
            S.nx = nx;
            S.ny = ny;
            S.bc = b->cfg.boundary;
            S.cu = cu;
            S.nlags = nlags;
            S.p = p;
            S.partial = part;
            r = launch_structure_sweep(pi, dim3(cu + ct, nlags, m), b->stream, S);
        } else {
            r = launch_structure_gather(pi, dim3(cu, nlags, m), b->stream, state, stride, var, nx, ny, b->dim,
                                        b->cfg.boundary, p, part);
        }
        if (r) return r;
        const double factor = b->dim == 2 && b->cfg.boundary == AVH_BC_PERIODIC ? 2.0 : 1.0;
        hipLaunchKernelGGL(structure_finish_kernel, dim3((m * number_of_h + 3) / 4), dim3(256), 0, b->stream, part,
                           cu + ct, number_of_h, m, (double)G.ncells, factor, d);
        AVH_HIP(hipGetLastError());
        AVH_HIP(hipMemcpyAsync(out + (size_t)s0 * number_of_h, d, sizeof(double) * m * number_of_h,
                               hipMemcpyDeviceToHost, b->stream));
        AVH_HIP(hipStreamSynchronize(b->stream));
    }
    return AVH_OK;
}

avh_status avh_batch_set_tile_shape(avh_batch* b, int shape) {
    if (!b) return fail(AVH_EINVAL, "null argument");
    if (shape < -1 || shape >= num_shapes(b->dim)) return fail(AVH_EINVAL, "no such tile shape");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    b->graph.reset();
    b->shape = shape;
    return AVH_OK;
}

avh_status avh_batch_autotune(avh_batch* b, int* best_shape, double* ms_per_shape, int* nshapes) {
    if (!b) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(b->device));
    return batch_autotune(b, best_shape, ms_per_shape, nshapes);
}

avh_status avh_batch_time_step_kernels(avh_batch* b, int64_t steps, double* ms, int* kernels) {
    if (!b || !ms || !kernels || steps < 1 || steps > 100000) return fail(AVH_EINVAL, "bad argument");
    AVH_HIP(hipSetDevice(b->device));
    const int nk = batch_launches_per_step(b);
    avh_status r = batch_ensure_shape(b);
    if (r) return r;
    EventMarks t;
    if ((r = t.create((size_t)steps * (nk + 1)))) return r;
    for (int64_t k = 0; k < steps; ++k)
        if ((r = enqueue_batch_step(b, &t))) return r;
    if ((r = t.average(steps, nk, ms))) return r;
    *kernels = nk;
    return AVH_OK;
}

avh_status avh_batch_get_progress(avh_batch* b, int group, int sample, avh_progress* p) {
    avh_status r = check_gs(b, group, sample);
    if (r) return r;
    if (!p) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    Control c;
    AVH_HIP(hipMemcpy(&c, b->g[group].ctrl + sample, sizeof c, hipMemcpyDeviceToHost));
    p->time = c.t;
    p->last_dt = c.last_dt;
    p->steps = c.steps;
    p->violated = c.violated;
    p->saves_pending = c.saves_pending;
    return AVH_OK;
}

avh_status avh_batch_get_statistics(avh_batch* b, int group, int save, int primitive, double* mean,
                                    double* variance, int64_t* count) {
    avh_status r = check_gs(b, group, 0);
    if (r) return r;
    if (!mean || !variance || !count) return fail(AVH_EINVAL, "null argument");
    if (save < 0 || save >= b->nsaves) return fail(AVH_EINVAL, "no such statistics save");
    AVH_HIP(hipSetDevice(b->device));
    AVH_HIP(hipStreamSynchronize(b->stream));
    const GroupHost& G = b->g[group];
    const size_t n = (size_t)b->nv * G.ncells;
    const size_t off = (size_t)save * n;
    long long cnt = 0;
    AVH_HIP(hipMemcpy(&cnt, G.counts + save, sizeof cnt, hipMemcpyDeviceToHost));
    AVH_HIP(hipMemcpy(mean, (primitive ? G.mean_p : G.mean_c) + off, n * sizeof(double), hipMemcpyDeviceToHost));
    AVH_HIP(hipMemcpy(variance, (primitive ? G.m2_p : G.m2_c) + off, n * sizeof(double), hipMemcpyDeviceToHost));
    // population variance M2 / M (the reference's M2/M - mean^2,
    // alsuq/src/stats/MeanVariance.cpp:55-67, StatisticsHelper.cpp:70-72)
    for (size_t i = 0; i < n; ++i) variance[i] = cnt > 0 ? variance[i] / (double)cnt : 0.0;
    *count = cnt;
    return AVH_OK;
}

avh_status avh_uq_generate(int nparams, const int* dims, const double* lower, const double* upper,
                           int64_t sample_start, int64_t nsamples, double* out) {
    if (nparams < 1 || !dims || !lower || !upper || !out || sample_start < 0 || nsamples < 0)
        return fail(AVH_EINVAL, "bad argument");
    // One default-seeded std::mt19937_64 shared by every parameter, with the
    // reference's fast-forward: component c of sample s of a parameter of
    // dimension D is preceded by s*D + c draws counted on the shared counter
    // (alsuq/src/generator/STLMersenne.cpp:25-85); uniform_real_distribution
    // <double>(0,1) scaled to [lower, upper) (alsuq/src/distribution/
    // Uniform.cpp:27-34); parameters in the caller's order, which is the
    // reference's parameter-name order.
    std::mt19937_64 engine;
    long counter = 0;
    std::uniform_real_distribution<double> dist(0.0, 1.0);
    size_t o = 0;
    for (int64_t s = sample_start; s < sample_start + nsamples; ++s) {
        for (int p = 0; p < nparams; ++p) {
            const long dimension = dims[p];
            if (dimension < 1) return fail(AVH_EINVAL, "parameter dimensions must be >= 1");
            for (long c = 0; c < dimension; ++c) {
                if (counter / dimension < long(s)) {
                    const long add = long(s) * dimension - counter;
                    engine.discard(add);
                    counter += add;
                }
                if (counter % dimension < c) {
                    const long add = c - counter % dimension;
                    engine.discard(add);
                    counter += add;
                }
                counter++;
                const double x = dist(engine);
                out[o++] = x * (upper[p] - lower[p]) + lower[p];
            }
        }
    }
    return AVH_OK;
}

}  // extern "C"
