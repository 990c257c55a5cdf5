// Surrogate network of the hip platform: an ensemble of multilayer
// perceptrons (inputs -> hidden GELU layers -> outputs) trained with Adam,
// every member in the same launches (blockIdx.z = member).
//
// Arithmetic: weights, activations and backward signals are stored in bf16;
// every product runs on the matrix cores (v_mfma_f32_16x16x32_bf16, with one 16x16x16 step for a K tail of 16) with
// fp32 accumulation; biases, pre-activations, outputs, gradients and the
// Adam state are fp32.  Feature dimensions are padded to multiples of 16
// with zeros (the padded weights get zero gradients and stay zero).
//
// All products are written C[m][n] = sum_k A[m][k] * B[n][k] with both
// operands k-contiguous, so activations are kept in both orientations:
//   forward   Z_l  = X_l  . W_l^T + b_l,   X_{l+1} = gelu(Z_l)
//   backward  dW_l = dZ_l^T . X_l           (operands dZ_l^T, X_l^T)
//             dX_l = dZ_l . W_l             (operands dZ_l, W_l^T)
//             dZ_{l-1} = dX_l * gelu'(Z_{l-1})
// Networks whose layers fit a workgroup's LDS (FUSED_MAX_DIM) run a training
// step in two launches -- mlp_rows_kernel takes 16 rows through every layer
// and back, mlp_update_kernel forms all gradients and applies Adam -- and a
// prediction in one; wider ones run layer by layer (mlp_gemm_kernel).  Both
// form every product with the same matrix instructions in the same order.
// No reference counterpart: the reference has no learned model; this is the
// surrogate of its Monte Carlo runs (alsuq/src/run/Runner.cpp:39-90).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>
#include <random>
#include <vector>

#include "avh_internal.hpp"

using namespace avh;

namespace {

constexpr int MAX_LAYERS = 8;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
    // round to nearest even; NaN stays NaN
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// exact GELU, x * Phi(x), and its derivative Phi(x) + x * phi(x)
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}
// both from one erff: the same bits as gelu and gelu_grad
__device__ __forceinline__ float gelu_both(float x, float& grad) {
    const float e = 1.0f + erff(x * 0.70710678118654752f);
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    grad = 0.5f * e + x * pdf;
    return 0.5f * x * e;
}

enum GemmEpilogue { EPI_HIDDEN = 0, EPI_OUT = 1, EPI_DX = 2, EPI_DW = 3 };

struct GemmArgs {
    const uint16_t* A;  // [M][K] per member
    const uint16_t* B;  // [N][K] per member
    long long a_ms, b_ms;
    int lda, ldb;
    int M, N, K;
    const float* bias;  // [N] per member (EPI_HIDDEN / EPI_OUT)
    long long bias_ms;
    float* C32;         // [M][N] fp32 out: Z, outputs or dW
    long long c32_ms;
    uint16_t* Cb;       // [M][N] bf16 out: activations or dZ_prev
    uint16_t* CbT;      // [N][M] bf16 out, transposed
    long long cb_ms;
    const float* Zp;    // [M][N] pre-activations of the previous layer (EPI_DX)
    long long zp_ms;
};

// One wavefront per 16x16 tile of C, four per workgroup (32x32).  The whole
// wavefront skips a tile outside C, so the matrix instruction always runs
// with every lane active.
template <int EPI>
__global__ __launch_bounds__(256) void mlp_gemm_kernel(GemmArgs g) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int tm = blockIdx.y * 2 + (w >> 1), tn = blockIdx.x * 2 + (w & 1);
    if (tm * 16 >= g.M || tn * 16 >= g.N) return;
    const int mem = blockIdx.z;
    const uint16_t* A = g.A + mem * g.a_ms + (long long)(tm * 16 + (lane & 15)) * g.lda;
    const uint16_t* B = g.B + mem * g.b_ms + (long long)(tn * 16 + (lane & 15)) * g.ldb;
    const int kq = lane >> 4;  // the lane's quarter of each K step
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // K steps of 32 on gfx950's v_mfma_f32_16x16x32_bf16 (8 consecutive k
    // per lane, 16-byte loads), then a step of 16 for K = 16 mod 32 (the
    // padded widths 48 and 80)
    int k0 = 0;
    for (; k0 + 32 <= g.K; k0 += 32) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(A + k0 + 8 * kq);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(B + k0 + 8 * kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
    }
    if (k0 < g.K) {
        const bf16x4 a = *reinterpret_cast<const bf16x4*>(A + k0 + 4 * kq);
        const bf16x4 b = *reinterpret_cast<const bf16x4*>(B + k0 + 4 * kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    const int n = tn * 16 + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = tm * 16 + 4 * (lane >> 4) + r;
        const long long o = (long long)m * g.N + n;
        const long long ot = (long long)n * g.M + m;
        float v = acc[r];
        if (EPI == EPI_HIDDEN) {
            v += g.bias[mem * g.bias_ms + n];
            g.C32[mem * g.c32_ms + o] = v;
            const uint16_t a = f2bf(gelu(v));
            g.Cb[mem * g.cb_ms + o] = a;
            g.CbT[mem * g.cb_ms + ot] = a;
        } else if (EPI == EPI_OUT) {
            g.C32[mem * g.c32_ms + o] = v + g.bias[mem * g.bias_ms + n];
        } else if (EPI == EPI_DX) {
            const uint16_t d = f2bf(v * gelu_grad(g.Zp[mem * g.zp_ms + o]));
            g.Cb[mem * g.cb_ms + o] = d;
            g.CbT[mem * g.cb_ms + ot] = d;
        } else {
            g.C32[mem * g.c32_ms + o] = v;
        }
    }
}

// Minibatch rows: X0 = bf16((x - mean) / std) (both orientations), targets
// (y - mean) / std; rows past `rows` and padded features are zero.
__global__ __launch_bounds__(256) void mlp_gather_kernel(const float* X, const float* Y, const int* idx, long long idx_ms,
                                                         int rows, int nin, int pin, int nout, int pout, int B,
                                                         const float* in_mu, const float* in_sd, const float* out_mu,
                                                         const float* out_sd, uint16_t* X0, uint16_t* X0T, float* Yn) {
    const int mem = blockIdx.z;
    const int r = blockIdx.x;  // row of the minibatch
    const bool live = r < rows;
    const long long src = live ? (long long)idx[mem * idx_ms + r] : 0;
    for (int k = threadIdx.x; k < pin; k += blockDim.x) {
        float v = 0.f;
        if (live && k < nin) v = (X[src * nin + k] - in_mu[k]) / in_sd[k];
        const uint16_t b = f2bf(v);
        X0[((long long)mem * B + r) * pin + k] = b;
        X0T[((long long)mem * pin + k) * B + r] = b;
    }
    if (Y) {
        for (int o = threadIdx.x; o < pout; o += blockDim.x) {
            float v = 0.f;
            if (live && o < nout) v = (Y[src * nout + o] - out_mu[o]) / out_sd[o];
            Yn[((long long)mem * B + r) * pout + o] = v;
        }
    }
}

// Mean-squared error over the real outputs and its gradient
// 2 (yhat - y) / (B * nout) in both orientations; the loss of each member is
// added to loss[mem] (fixed-order tree, so it is reproducible).
__global__ __launch_bounds__(256) void mlp_loss_kernel(const float* Yhat, const float* Yn, int B, int nout, int pout,
                                                       uint16_t* dZ, uint16_t* dZT, long long dz_ms, float* loss) {
    __shared__ float red[256];
    const int mem = blockIdx.x;
    const float scale = 2.0f / (float)(B * nout);
    float acc = 0.f;
    for (int t = threadIdx.x; t < B * pout; t += 256) {
        const int r = t / pout, o = t % pout;
        const long long i = (long long)mem * B * pout + t;
        const float d = o < nout ? Yhat[i] - Yn[i] : 0.f;
        acc += d * d;
        const uint16_t g = f2bf(d * scale);
        dZ[mem * dz_ms + (long long)r * pout + o] = g;
        dZT[mem * dz_ms + (long long)o * B + r] = g;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss[mem] += red[0] / (float)(B * nout);
}

// db[o] = sum over the minibatch rows of dZ[r][o], in row order.
__global__ __launch_bounds__(256) void mlp_bias_grad_kernel(const uint16_t* dZT, long long dz_ms, int nout, int B,
                                                            float* grad, long long p_ms, long long b_off) {
    const int mem = blockIdx.y;
    const int o = blockIdx.x * 256 + threadIdx.x;
    if (o >= nout) return;
    const uint16_t* row = dZT + mem * dz_ms + (long long)o * B;
    float acc = 0.f;
    for (int r = 0; r < B; ++r) acc += bf2f(row[r]);
    grad[mem * p_ms + b_off + o] = acc;
}

// Tile layout of a 16-bit operand [rows][K] of the fused path (rows and K
// multiples of 16): 16 rows x 32 of K are 1 KiB in the order in which the
// lanes of a matrix instruction take them (lane = row % 16 + 16 * (k % 32 / 8),
// 8 values each), a last 16 of K likewise with 4 values a lane.  A wave's
// operand load is then one contiguous block; row-major rows of 512 bytes put
// its 64 lanes on 16 cache lines of the same banks (a 256-wide layer's weights
// took 9000 cycles to arrive, 2048 at L1's rate).
__host__ __device__ __forceinline__ int tiled(int row, int k, int K) {
    const int full = K & ~31, tile = (row >> 4) * 16 * K;
    if (k < full) return tile + (k >> 5) * 512 + ((k & 31) >> 3) * 128 + (row & 15) * 8 + (k & 7);
    return tile + full * 16 + ((k & 15) >> 2) * 64 + (row & 15) * 4 + (k & 3);
}

struct LayerDesc {
    int nin, nout;
    long long w_off, b_off;  // in the fp32 parameter block of a member
    long long wb_off;        // in the bf16 weight blocks of a member
};

struct AdamArgs {
    float *p, *m, *v;
    const float* g;
    uint16_t *wb, *wtb;
    long long p_ms, wb_ms;
    LayerDesc L[MAX_LAYERS];
    float lr, b1, b2, eps, c1, c2;  // c1 = 1 - b1^t, c2 = 1 - b2^t
    float wd;                       // decoupled weight decay of the weights (not the biases)
    int tiles;                      // bf16 weights in the fused path's tile layout
};

// where weight (o, k) of a layer goes in the bf16 blocks
__device__ __forceinline__ int weight_at(const AdamArgs& a, const LayerDesc& L, int o, int k) {
    return a.tiles ? tiled(o, k, L.nin) : o * L.nin + k;
}
__device__ __forceinline__ int weight_t_at(const AdamArgs& a, const LayerDesc& L, int o, int k) {
    return a.tiles ? tiled(k, o, L.nout) : k * L.nout + o;
}

// Adam's update of one parameter; writes p, m, v and returns the new value.
__device__ __forceinline__ float adam_update(const AdamArgs& a, long long i, float g, float p0, float m0, float v0,
                                             bool weight) {
    const float m = a.b1 * m0 + (1.f - a.b1) * g;
    const float v = a.b2 * v0 + (1.f - a.b2) * (g * g);
    a.m[i] = m;
    a.v[i] = v;
    float p = p0 - a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
    if (weight && a.wd != 0.f) p = p - a.lr * a.wd * p0;
    a.p[i] = p;
    return p;
}

// Adam (bias-corrected) on the fp32 master parameters of layer blockIdx.y,
// with decoupled weight decay on the weights (AdamW, Loshchilov and Hutter,
// "Decoupled Weight Decay Regularization", 2019: p -= lr * wd * p beside the
// Adam step), then the bf16 copies of the weights in both orientations.
__global__ __launch_bounds__(256) void mlp_adam_kernel(AdamArgs a) {
    const LayerDesc& L = a.L[blockIdx.y];
    const int mem = blockIdx.z;
    const long long nw = (long long)L.nin * L.nout;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= nw + L.nout) return;
    const long long i = mem * a.p_ms + (e < nw ? L.w_off + e : L.b_off + (e - nw));
    const float p = adam_update(a, i, a.g[i], a.p[i], a.m[i], a.v[i], e < nw);
    if (e < nw) {
        const int o = (int)(e / L.nin), k = (int)(e % L.nin);
        const uint16_t b = f2bf(p);
        a.wb[mem * a.wb_ms + L.wb_off + weight_at(a, L, o, k)] = b;
        a.wtb[mem * a.wb_ms + L.wb_off + weight_t_at(a, L, o, k)] = b;
    }
}

// bf16 copies of every weight after the host set the fp32 parameters.
__global__ __launch_bounds__(256) void mlp_cast_kernel(AdamArgs a) {
    const LayerDesc& L = a.L[blockIdx.y];
    const int mem = blockIdx.z;
    const long long nw = (long long)L.nin * L.nout;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= nw) return;
    const int o = (int)(e / L.nin), k = (int)(e % L.nin);
    const uint16_t b = f2bf(a.p[mem * a.p_ms + L.w_off + e]);
    a.wb[mem * a.wb_ms + L.wb_off + weight_at(a, L, o, k)] = b;
    a.wtb[mem * a.wb_ms + L.wb_off + weight_t_at(a, L, o, k)] = b;
}

// ---------------------------------------------------------------------------
// The fused step.  One Adam step of the study's ensemble (5 members, 256 rows,
// 40 -> 256^4 -> 66) is 1.7 GFLOP and was 22 dependent launches of 3 to 40 us:
// latency, not arithmetic, bounds it, so the layers' activations stay in one
// workgroup's LDS and the launches go (347 -> 40 us a step, of which
// mlp_rows_kernel 25 and mlp_update_kernel 14).

// Widest layer of a network that takes the fused path: its two activation
// buffers take 33 KB of LDS, and no measured shape up to it is faster layer
// by layer (us a training step, fused / layered: 5 members of 512 x 4, 256
// rows 122 / 387; of 256 x 4, 4096 rows 401 / 3660; 64 members of 512 x 4,
// 1024 rows 2802 / 6605).  Wider layers would need a larger share of LDS, and
// every workgroup reads all of a member's weights.
constexpr int FUSED_MAX_DIM = 512;
constexpr int ROWS = 16;  // minibatch rows of a workgroup: one MFMA tile

struct RowsArgs {
    const float *X, *Y;     // data rows
    const int* idx;         // [member] rows of the minibatch, null: rows in order
    long long idx_ms;
    int rows;               // rows there are (later rows of a tile are zero)
    int nin, pin, nout, pout, B, M, W, nl;
    int pitch;              // LDS elements from one row to the next
    const float *mu_in, *sd_in, *mu_out, *sd_out;
    const uint16_t *wb, *wtb;
    long long wb_ms;
    const float* params;
    long long p_ms;
    LayerDesc L[MAX_LAYERS];
    float* dg;              // [hidden][member][B][W] gelu' of the pre-activations
    uint16_t *x0t, *at;     // transposed activations, for the gradients (tile layout)
    uint16_t* dzt;          // [layer][member][dz_w][B] transposed dZ (tile layout)
    int dz_w;
    float* loss_part;       // [member][workgroup]
    float* out;             // prediction: [member][rows][nout], data units
};

// bf16 by the hardware's conversion (round to nearest even, as f2bf)
__device__ __forceinline__ uint16_t cvt_bf(float f) {
    const __bf16 b = (__bf16)f;
    uint16_t u;
    __builtin_memcpy(&u, &b, 2);
    return u;
}

// One 16 x 16 tile of C = A . B^T: A's rows from LDS, B's tile (in tile
// layout) from global memory.  Of a K of 256 or more the first 256 of B are
// loaded ahead (load_ahead) and run without a branch; the steps' order is
// mlp_gemm_kernel's.
constexpr int AHEAD = 8;
__device__ __forceinline__ bf16x8 load8(const uint16_t* tile, int k0, int lane) {
    return *reinterpret_cast<const bf16x8*>(tile + k0 * 16 + lane * 8);
}
__device__ __forceinline__ bf16x4 load4(const uint16_t* tile, int k0, int lane) {
    return *reinterpret_cast<const bf16x4*>(tile + k0 * 16 + lane * 4);
}
__device__ __forceinline__ void load_ahead(const uint16_t* tile, int K, int lane, bf16x8 (&wreg)[AHEAD]) {
    if (K >= AHEAD * 32) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) wreg[i] = load8(tile, i * 32, lane);
    }
}
__device__ __forceinline__ f32x4 tile_product(const uint16_t* A, const uint16_t* tile, int K, int lane,
                                              const bf16x8 (&wreg)[AHEAD]) {
    const int kq = lane >> 4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int k0 = 0;
    if (K >= AHEAD * 32) {
        bf16x8 a[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) a[i] = *reinterpret_cast<const bf16x8*>(A + i * 32 + 8 * kq);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], wreg[i], acc, 0, 0, 0);
        k0 = AHEAD * 32;
    }
#pragma unroll 2
    for (; k0 + 32 <= K; k0 += 32) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(A + k0 + 8 * kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, load8(tile, k0, lane), acc, 0, 0, 0);
    }
    if (k0 < K) {
        const bf16x4 a = *reinterpret_cast<const bf16x4*>(A + k0 + 4 * kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, load4(tile, k0, lane), acc, 0, 0, 0);
    }
    return acc;
}

__device__ __forceinline__ void store4(uint16_t* to, const uint16_t (&v)[4]) {
    uint2 w;
    w.x = (uint32_t)v[0] | ((uint32_t)v[1] << 16);
    w.y = (uint32_t)v[2] | ((uint32_t)v[3] << 16);
    *reinterpret_cast<uint2*>(to) = w;
}

// Workgroup (x, member) takes ROWS rows through every layer, its waves sharing
// the layer's 16-column tiles; with TRAIN on to the loss and back to dZ of
// every layer.  Activations and backward signals alternate between two LDS
// buffers, one barrier a layer; a row's pitch is 16 bytes past a multiple of
// 32, so that the rows of a tile start in different banks.  TRAIN leaves what
// the gradients need (transposed activations and dZ) in global memory: a lane
// holds four consecutive rows of a column, one 8-byte store.  A wave loads its
// tile's weights, bias and gelu' of the next layer before it issues those
// stores: vector memory completes in order, and loads behind the stores would
// wait for them in every layer.  GELU and its derivative, an erff and an expf,
// are the longest part of a layer's chain and are formed together, forward.
// (5 members x 256 rows: 25 us in 80 workgroups; with the weights in rows
// 38 us; 160 workgroups of 8 rows, each wave with two tiles, 26 us.)
template <bool TRAIN>
__global__ __launch_bounds__(1024) void mlp_rows_kernel(RowsArgs g) {
    extern __shared__ __align__(16) uint16_t lds[];
    __shared__ int s_src[ROWS];
    __shared__ float s_loss[16];
    uint16_t* cur = lds;
    uint16_t* nxt = lds + ROWS * g.pitch;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int kq = lane >> 4, lo = lane & 15;
    const int mr = 4 * kq;  // the lane's first row of a result tile
    const int mem = blockIdx.y;
    const int row0 = blockIdx.x * ROWS;
    const uint16_t* wb = g.wb + mem * g.wb_ms;
    const uint16_t* wtb = g.wtb + mem * g.wb_ms;
    const float* params = g.params + mem * g.p_ms;
    // Every wave takes a 16-column tile of each product (waves past the last
    // repeat it and write the same values), so the code below has no branch
    // around its loads and stores; further tiles follow in a loop.
    auto first_tile = [&](int N) { return wave < N / 16 ? wave : N / 16 - 1; };
    bf16x8 wreg[AHEAD];
    auto product = [&](const uint16_t* W, int t, int K) {
        return tile_product(cur + lo * g.pitch, W + t * 16 * K, K, lane, wreg);
    };
    float bn = 0.f;  // the lane's bias in the next layer
    auto next_layer = [&](int l) {
        const LayerDesc L = g.L[l];
        const int t = first_tile(L.nout);
        load_ahead(wb + L.wb_off + t * 16 * L.nin, L.nin, lane, wreg);
        bn = params[L.b_off + t * 16 + lo];
    };
    float dg[4] = {0.f, 0.f, 0.f, 0.f};  // and gelu' in the next layer back
    auto dg_rows = [&](int l) { return g.dg + (((long long)l * g.M + mem) * g.B + row0 + mr) * g.W; };
    auto next_back = [&](int l) {
        const LayerDesc L = g.L[l];
        const int t = first_tile(L.nin);
        load_ahead(wtb + L.wb_off + t * 16 * L.nout, L.nout, lane, wreg);
        const float* d = dg_rows(l - 1) + t * 16 + lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) dg[r] = d[r * g.W];
    };
    auto swap = [&]() {
        lds_barrier();
        uint16_t* const sw = cur;
        cur = nxt;
        nxt = sw;
    };
    next_layer(0);

    if (threadIdx.x < ROWS) {
        const int r = row0 + threadIdx.x;
        s_src[threadIdx.x] = r < g.rows ? (g.idx ? g.idx[mem * g.idx_ms + r] : r) : -1;
    }
    lds_barrier();
    for (int e = threadIdx.x; e < ROWS * g.pin; e += blockDim.x) {
        const int r = e / g.pin, k = e % g.pin;
        const int src = s_src[r];
        float v = 0.f;
        if (src >= 0 && k < g.nin) v = (g.X[(long long)src * g.nin + k] - g.mu_in[k]) / g.sd_in[k];
        cur[r * g.pitch + k] = cvt_bf(v);
    }
    // normalised targets; those of the wave's output turn are loaded now
    auto target = [&](int m, int n) {
        const int src = s_src[m];
        return src >= 0 && n < g.nout ? (g.Y[(long long)src * g.nout + n] - g.mu_out[n]) / g.sd_out[n] : 0.f;
    };
    float y[4] = {0.f, 0.f, 0.f, 0.f};
    if (TRAIN) {
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = target(mr + r, first_tile(g.pout) * 16 + lo);
    }
    lds_barrier();
    if (TRAIN) {
        for (int e = threadIdx.x; e < 4 * g.pin; e += blockDim.x) {
            const int k = e >> 2, r = (e & 3) * 4;
            uint16_t q[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) q[i] = cur[(r + i) * g.pitch + k];
            store4(g.x0t + (long long)mem * g.pin * g.B + tiled(k, row0 + r, g.B), q);
        }
    }

    // hidden layers
    for (int l = 0; l + 1 < g.nl; ++l) {
        const LayerDesc L = g.L[l];
        const int N = L.nout;
        uint16_t* at = g.at + ((long long)l * g.M + mem) * g.W * g.B;
        float* dgl = dg_rows(l);
        uint16_t q[4];
        float grad[4];
        auto activate = [&](const f32x4& acc, int n, float b) {
#pragma unroll
            for (int r = 0; r < 4; ++r) q[r] = cvt_bf(TRAIN ? gelu_both(acc[r] + b, grad[r]) : gelu(acc[r] + b));
#pragma unroll
            for (int r = 0; r < 4; ++r) nxt[(mr + r) * g.pitch + n] = q[r];
        };
        auto keep = [&](int n) {
            if (!TRAIN) return;
#pragma unroll
            for (int r = 0; r < 4; ++r) dgl[r * g.W + n] = grad[r];
            store4(at + tiled(n, row0 + mr, g.B), q);
        };
        const uint16_t* W = wb + L.wb_off;
        const f32x4 acc = product(W, first_tile(N), L.nin);
        const float b = bn;
        for (int t = wave + nw; t < N / 16; t += nw) {
            load_ahead(W + t * 16 * L.nin, L.nin, lane, wreg);
            const int n = t * 16 + lo;
            activate(product(W, t, L.nin), n, params[L.b_off + n]);
            keep(n);
        }
        const int n = first_tile(N) * 16 + lo;
        activate(acc, n, b);
        next_layer(l + 1);
        keep(n);
        swap();
    }

    // output layer
    float loss = 0.f;
    {
        const int l = g.nl - 1;
        const LayerDesc L = g.L[l];
        const int N = L.nout;
        const uint16_t* W = wb + L.wb_off;
        const float scale = 2.0f / (float)(g.B * g.nout);
        uint16_t* dzt = g.dzt + ((long long)l * g.M + mem) * g.dz_w * g.B;
        uint16_t q[4];
        auto finish = [&](const f32x4& acc, int t, float b) {
            const int n = t * 16 + lo;
            if (TRAIN) {
                const bool own = t == wave || t >= nw;  // not a repeat
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = acc[r] + b;
                    const float d = n < g.nout ? v - (t < nw ? y[r] : target(mr + r, n)) : 0.f;
                    loss += own ? d * d : 0.f;
                    q[r] = cvt_bf(d * scale);
                    nxt[(mr + r) * g.pitch + n] = q[r];
                }
            } else if (n < g.nout) {
                const float sd = g.sd_out[n], mu = g.mu_out[n];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row0 + mr + r < g.rows)
                        g.out[((long long)mem * g.rows + row0 + mr + r) * g.nout + n] = (acc[r] + b) * sd + mu;
            }
        };
        const f32x4 acc = product(W, first_tile(N), L.nin);
        for (int t = wave + nw; t < N / 16; t += nw) {
            load_ahead(W + t * 16 * L.nin, L.nin, lane, wreg);
            finish(product(W, t, L.nin), t, params[L.b_off + t * 16 + lo]);
            if (TRAIN) store4(dzt + tiled(t * 16 + lo, row0 + mr, g.B), q);
        }
        finish(acc, first_tile(N), bn);
        if (!TRAIN) return;
        next_back(l);
        store4(dzt + tiled(first_tile(N) * 16 + lo, row0 + mr, g.B), q);
        swap();
    }

    // dZ_{l-1} = (dZ_l . W_l) * gelu'(Z_{l-1})
    for (int l = g.nl - 1; l > 0; --l) {
        const LayerDesc L = g.L[l];
        const int K = L.nout, N = L.nin;
        const uint16_t* W = wtb + L.wb_off;
        uint16_t* dzt = g.dzt + ((long long)(l - 1) * g.M + mem) * g.dz_w * g.B;
        uint16_t q[4];
        auto finish = [&](const f32x4& acc, int n, const float (&d)[4]) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                q[r] = cvt_bf(acc[r] * d[r]);
                nxt[(mr + r) * g.pitch + n] = q[r];
            }
        };
        const f32x4 acc = product(W, first_tile(N), K);
        for (int t = wave + nw; t < N / 16; t += nw) {
            load_ahead(W + t * 16 * K, K, lane, wreg);
            const int n = t * 16 + lo;
            float d[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) d[r] = dg_rows(l - 1)[r * g.W + n];
            finish(product(W, t, K), n, d);
            store4(dzt + tiled(n, row0 + mr, g.B), q);
        }
        const int n = first_tile(N) * 16 + lo;
        finish(acc, n, dg);
        if (l > 1) next_back(l - 1);
        store4(dzt + tiled(n, row0 + mr, g.B), q);
        swap();
    }

    // the workgroup's share of the loss, the same tree every time
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) s_loss[wave] = loss;
    lds_barrier();
    if (threadIdx.x == 0) {
        float sum = 0.f;
        for (int w = 0; w < nw; ++w) sum += s_loss[w];
        g.loss_part[(long long)mem * gridDim.x + blockIdx.x] = sum;
    }
}

struct UpdateArgs {
    AdamArgs a;
    float* grad;
    const uint16_t *x0t, *at, *dzt;
    int pin, W, B, M, nl, dz_w, nout;
    int bias_blocks;            // workgroups of the biases, the first ones
    int first[MAX_LAYERS + 1];  // first workgroup of each layer's weights among the others, and their number
    const float* loss_part;
    int nparts;
    float* loss;
};

// Gradients of every layer, dW = dZ^T . X over the minibatch rows and db in
// row order, with Adam on the spot (ADAM) and the bf16 copies of the weights.
// Bound by the latency of its operands in L2 and of the master weights and
// moments in HBM; a wave takes a 16 x 32 tile of dW, whose moments and weights
// it loads before the products.  The first workgroups sum the biases (one lane
// an output: a chain of B additions, the longest work here) and the loss.
template <bool ADAM>
__global__ __launch_bounds__(256) void mlp_update_kernel(UpdateArgs u) {
    const AdamArgs& a = u.a;
    const int mem = blockIdx.y, part = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (part >= u.bias_blocks) {
        const int b = part - u.bias_blocks;
        // the layer, selected from all of the table: a search step by step
        // would wait for a scalar load at every step
        int l = 0, first = 0;
        LayerDesc L = a.L[0];
#pragma unroll
        for (int i = 1; i < MAX_LAYERS; ++i)
            if (i < u.nl && b >= u.first[i]) {
                l = i;
                first = u.first[i];
                L = a.L[i];
            }
        const int ntn = (L.nin + 31) / 32;
        const int tile = (b - first) * 4 + wave;
        const int tm = tile / ntn, tn = tile % ntn;
        if (tm * 16 >= L.nout) return;
        const int kq = lane >> 4, lo = lane & 15;
        const uint16_t* A = u.dzt + (((long long)l * u.M + mem) * u.dz_w + tm * 16) * u.B;
        const uint16_t* X = l == 0 ? u.x0t + (long long)mem * u.pin * u.B
                                   : u.at + ((long long)(l - 1) * u.M + mem) * u.W * u.B;
        const bool two = tn * 32 + 16 < L.nin;  // the second half of the tile exists
        const int n[2] = {tn * 32 + lo, two ? tn * 32 + 16 + lo : tn * 32 + lo};
        long long at[2][4];
        float p0[2][4], m0[2][4], v0[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                at[h][r] = mem * a.p_ms + L.w_off + (long long)(tm * 16 + 4 * kq + r) * L.nin + n[h];
                if (ADAM) {
                    p0[h][r] = a.p[at[h][r]];
                    m0[h][r] = a.m[at[h][r]];
                    v0[h][r] = a.v[at[h][r]];
                }
            }
        const uint16_t* X0 = X + tn * 32 * u.B;
        const uint16_t* X1 = two ? X0 + 16 * u.B : X0;
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        int k0 = 0;
#pragma unroll 4
        for (; k0 + 32 <= u.B; k0 += 32) {
            const bf16x8 x = load8(A, k0, lane), y0 = load8(X0, k0, lane), y1 = load8(X1, k0, lane);
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y0, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y1, acc[1], 0, 0, 0);
        }
        if (k0 < u.B) {
            const bf16x4 x = load4(A, k0, lane), y0 = load4(X0, k0, lane), y1 = load4(X1, k0, lane);
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, y0, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, y1, acc[1], 0, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h == 1 && !two) break;
            uint16_t q[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float g = acc[h][r];
                u.grad[at[h][r]] = g;
                if (ADAM) {
                    q[r] = cvt_bf(adam_update(a, at[h][r], g, p0[h][r], m0[h][r], v0[h][r], true));
                    a.wb[mem * a.wb_ms + L.wb_off + tiled(tm * 16 + 4 * kq + r, n[h], L.nin)] = q[r];
                }
            }
            if (ADAM) store4(a.wtb + mem * a.wb_ms + L.wb_off + tiled(n[h], tm * 16 + 4 * kq, L.nout), q);
        }
        return;
    }
    // biases: output t of all layers in turn, a lane each
    int t = part * 256 + threadIdx.x;
    if (t == 0) {
        float sum = 0.f;
        for (int i = 0; i < u.nparts; ++i) sum += u.loss_part[(long long)mem * u.nparts + i];
        u.loss[mem] += sum / (float)(u.B * u.nout);
    }
    int l = -1, at = 0;
    long long b_off = 0;
#pragma unroll
    for (int i = 0, base = 0; i < MAX_LAYERS; ++i)
        if (i < u.nl) {
            if (t >= base && t < base + a.L[i].nout) {
                l = i;
                at = base;
                b_off = a.L[i].b_off;
            }
            base += a.L[i].nout;
        }
    if (l < 0) return;
    t -= at;
    const uint16_t* dz = u.dzt + ((long long)l * u.M + mem) * u.dz_w * u.B;
    const long long i = mem * a.p_ms + b_off + t;
    float acc = 0.f;
#pragma unroll 8
    for (int r = 0; r < u.B; r += 4) {
        const uint2 w = *reinterpret_cast<const uint2*>(dz + tiled(t, r, u.B));
        acc += __uint_as_float(w.x << 16);
        acc += __uint_as_float(w.x & 0xffff0000u);
        acc += __uint_as_float(w.y << 16);
        acc += __uint_as_float(w.y & 0xffff0000u);
    }
    u.grad[i] = acc;
    if (ADAM) adam_update(a, i, acc, a.p[i], a.m[i], a.v[i], false);
}

// The fp32 block of a member (parameters or gradients) in the caller's order:
// W[out][in] without padding, then b[out], layer by layer.
struct PackArgs {
    const float* src;
    float* dst;
    long long src_ms, dst_ms;
    LayerDesc L[MAX_LAYERS];
    int fin[MAX_LAYERS], fout[MAX_LAYERS];  // unpadded widths
    long long off[MAX_LAYERS];              // layer's first value in the caller's order
};
__global__ __launch_bounds__(256) void mlp_pack_kernel(PackArgs a) {
    const int l = blockIdx.y, mem = blockIdx.z;
    const long long nw = (long long)a.fin[l] * a.fout[l];
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= nw + a.fout[l]) return;
    const LayerDesc& L = a.L[l];
    const long long i = e < nw ? L.w_off + e / a.fin[l] * L.nin + e % a.fin[l] : L.b_off + (e - nw);
    a.dst[mem * a.dst_ms + a.off[l] + e] = a.src[mem * a.src_ms + i];
}

inline int pad16(int x) { return (x + 15) / 16 * 16; }

}  // namespace

struct avh_mlp {
    int device = 0;
    avh_mlp_config cfg{};
    int nl = 0, pin = 0, pout = 0, B = 0, M = 0, maxw = 0;
    LayerDesc L[MAX_LAYERS];
    long long P = 0, WB = 0;
    float *params = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;
    uint16_t *wb = nullptr, *wtb = nullptr;
    uint16_t *x0t = nullptr, *at = nullptr;  // transposed inputs and activations
    float* z = nullptr;        // [hidden][M][B][width] pre-activations, or gelu' of them (fused)
    // of the layer-by-layer path alone
    uint16_t *x0 = nullptr, *a = nullptr;
    float *yhat = nullptr, *yn = nullptr;
    uint16_t *dz[2] = {nullptr, nullptr}, *dzt[2] = {nullptr, nullptr};
    float *mu_in = nullptr, *sd_in = nullptr, *mu_out = nullptr, *sd_out = nullptr;
    float* loss = nullptr;
    float *dx = nullptr, *dy = nullptr;
    long long dcap = 0;
    int* idx = nullptr;
    long long icap = 0;
    long long t = 0;  // Adam steps taken
    bool fused = false;         // the fused path serves this network
    uint16_t* dztl = nullptr;   // [layer][M][dz_w][B] transposed dZ (fused)
    float* loss_part = nullptr; // [M][row tiles] (fused)
    float* outbuf = nullptr;    // what a call hands to the host: predictions, packed parameters
    long long ocap = 0;
    long long epochs_done = 0;  // epochs of avh_mlp_train so far (seeds the shuffles)
    float wd = 0.f;   // decoupled weight decay
    hipStream_t stream = nullptr;
};

namespace {

void free_mlp(avh_mlp* n) {
    if (!n) return;
    (void)hipSetDevice(n->device);
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    void* ptrs[] = {n->params, n->m, n->v, n->grad, n->wb, n->wtb, n->x0, n->x0t, n->z, n->a, n->at, n->yhat,
                    n->yn, n->dz[0], n->dz[1], n->dzt[0], n->dzt[1], n->mu_in, n->sd_in, n->mu_out, n->sd_out,
                    n->loss, n->dx, n->dy, n->idx, n->dztl, n->loss_part, n->outbuf};
    for (void* p : ptrs) (void)hipFree(p);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

AdamArgs adam_args(const avh_mlp* n) {
    AdamArgs a;
    std::memset(&a, 0, sizeof a);
    a.p = n->params;
    a.m = n->m;
    a.v = n->v;
    a.g = n->grad;
    a.wb = n->wb;
    a.wtb = n->wtb;
    a.p_ms = n->P;
    a.wb_ms = n->WB;
    a.tiles = n->fused ? 1 : 0;
    for (int l = 0; l < n->nl; ++l) a.L[l] = n->L[l];
    return a;
}

unsigned int max_layer_blocks(const avh_mlp* n) {
    long long mx = 0;
    for (int l = 0; l < n->nl; ++l) mx = std::max(mx, (long long)n->L[l].nin * n->L[l].nout + n->L[l].nout);
    return (unsigned int)((mx + 255) / 256);
}

avh_status cast_weights(avh_mlp* n) {
    AdamArgs a = adam_args(n);
    hipLaunchKernelGGL(mlp_cast_kernel, dim3(max_layer_blocks(n), n->nl, n->M), dim3(256), 0, n->stream, a);
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

avh_status ensure_data(avh_mlp* n, long long rows) {
    if (rows <= n->dcap) return AVH_OK;
    (void)hipFree(n->dx);
    (void)hipFree(n->dy);
    n->dx = n->dy = nullptr;
    n->dcap = 0;
    AVH_HIP(hipMalloc(&n->dx, sizeof(float) * rows * n->cfg.n_in));
    AVH_HIP(hipMalloc(&n->dy, sizeof(float) * rows * n->cfg.n_out));
    n->dcap = rows;
    return AVH_OK;
}

avh_status ensure_idx(avh_mlp* n, long long count) {
    if (count <= n->icap) return AVH_OK;
    (void)hipFree(n->idx);
    n->idx = nullptr;
    n->icap = 0;
    AVH_HIP(hipMalloc(&n->idx, sizeof(int) * count));
    n->icap = count;
    return AVH_OK;
}

template <int EPI>
avh_status gemm(avh_mlp* n, const GemmArgs& g) {
    const dim3 grid((g.N + 31) / 32, (g.M + 31) / 32, n->M);
    hipLaunchKernelGGL(mlp_gemm_kernel<EPI>, grid, dim3(256), 0, n->stream, g);
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

// rows of the minibatch from the device data through idx[mem][row0 ...]
avh_status gather(avh_mlp* n, long long row0, long long idx_ms, int rows, bool targets) {
    hipLaunchKernelGGL(mlp_gather_kernel, dim3(n->B, 1, n->M), dim3(64), 0, n->stream, n->dx,
                       targets ? n->dy : nullptr, n->idx + row0, idx_ms, rows, n->cfg.n_in, n->pin,
                       n->cfg.n_out, n->pout, n->B, n->mu_in, n->sd_in, n->mu_out, n->sd_out, n->x0, n->x0t,
                       n->yn);
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

avh_status forward(avh_mlp* n) {
    const int H = n->nl - 1, W = n->maxw, B = n->B;
    for (int l = 0; l < n->nl; ++l) {
        const LayerDesc& L = n->L[l];
        GemmArgs g;
        std::memset(&g, 0, sizeof g);
        if (l == 0) {
            g.A = n->x0;
            g.a_ms = (long long)B * n->pin;
        } else {
            g.A = n->a + (long long)(l - 1) * n->M * B * W;
            g.a_ms = (long long)B * W;
        }
        g.lda = L.nin;
        g.B = n->wb + L.wb_off;
        g.b_ms = n->WB;
        g.ldb = L.nin;
        g.M = B;
        g.N = L.nout;
        g.K = L.nin;
        g.bias = n->params + L.b_off;
        g.bias_ms = n->P;
        if (l < H) {
            g.C32 = n->z + (long long)l * n->M * B * W;
            g.c32_ms = (long long)B * W;
            g.Cb = n->a + (long long)l * n->M * B * W;
            g.CbT = n->at + (long long)l * n->M * B * W;
            g.cb_ms = (long long)B * W;
            avh_status r = gemm<EPI_HIDDEN>(n, g);
            if (r) return r;
        } else {
            g.C32 = n->yhat;
            g.c32_ms = (long long)B * n->pout;
            avh_status r = gemm<EPI_OUT>(n, g);
            if (r) return r;
        }
    }
    return AVH_OK;
}

// Loss, gradients of every parameter into n->grad (no update).
avh_status backward(avh_mlp* n) {
    const int H = n->nl - 1, W = n->maxw, B = n->B;
    const long long dz_ms = (long long)B * std::max(W, n->pout);
    hipLaunchKernelGGL(mlp_loss_kernel, dim3(n->M), dim3(256), 0, n->stream, n->yhat, n->yn, B, n->cfg.n_out,
                       n->pout, n->dz[0], n->dzt[0], dz_ms, n->loss);
    AVH_HIP(hipGetLastError());
    int cur = 0;
    for (int l = n->nl - 1; l >= 0; --l) {
        const LayerDesc& L = n->L[l];
        // dW_l = dZ_l^T . X_l
        GemmArgs g;
        std::memset(&g, 0, sizeof g);
        g.A = n->dzt[cur];
        g.a_ms = dz_ms;
        g.lda = B;
        if (l == 0) {
            g.B = n->x0t;
            g.b_ms = (long long)n->pin * B;
        } else {
            g.B = n->at + (long long)(l - 1) * n->M * B * W;
            g.b_ms = (long long)W * B;
        }
        g.ldb = B;
        g.M = L.nout;
        g.N = L.nin;
        g.K = B;
        g.C32 = n->grad + L.w_off;
        g.c32_ms = n->P;
        avh_status r = gemm<EPI_DW>(n, g);
        if (r) return r;
        hipLaunchKernelGGL(mlp_bias_grad_kernel, dim3((L.nout + 255) / 256, n->M), dim3(256), 0, n->stream,
                           n->dzt[cur], dz_ms, L.nout, B, n->grad, n->P, L.b_off);
        AVH_HIP(hipGetLastError());
        if (l == 0) break;
        // dZ_{l-1} = (dZ_l . W_l) * gelu'(Z_{l-1})
        GemmArgs d;
        std::memset(&d, 0, sizeof d);
        d.A = n->dz[cur];
        d.a_ms = dz_ms;
        d.lda = L.nout;
        d.B = n->wtb + L.wb_off;
        d.b_ms = n->WB;
        d.ldb = L.nout;
        d.M = B;
        d.N = L.nin;
        d.K = L.nout;
        d.Zp = n->z + (long long)(l - 1) * n->M * B * W;
        d.zp_ms = (long long)B * W;
        d.Cb = n->dz[1 - cur];
        d.CbT = n->dzt[1 - cur];
        d.cb_ms = dz_ms;
        if ((r = gemm<EPI_DX>(n, d))) return r;
        cur = 1 - cur;
    }
    (void)H;
    return AVH_OK;
}

// Adam's arguments for the next step (counts it)
AdamArgs next_adam(avh_mlp* n, float lr) {
    n->t += 1;
    AdamArgs a = adam_args(n);
    a.lr = lr;
    a.wd = n->wd;
    a.b1 = n->cfg.beta1;
    a.b2 = n->cfg.beta2;
    a.eps = n->cfg.eps;
    a.c1 = (float)(1.0 - std::pow((double)n->cfg.beta1, (double)n->t));
    a.c2 = (float)(1.0 - std::pow((double)n->cfg.beta2, (double)n->t));
    return a;
}

avh_status adam_step(avh_mlp* n, float lr) {
    const AdamArgs a = next_adam(n, lr);
    hipLaunchKernelGGL(mlp_adam_kernel, dim3(max_layer_blocks(n), n->nl, n->M), dim3(256), 0, n->stream, a);
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

int dz_width(const avh_mlp* n) { return std::max(n->maxw, n->pout); }

RowsArgs rows_args(const avh_mlp* n) {
    RowsArgs g;
    std::memset(&g, 0, sizeof g);
    g.X = n->dx;
    g.nin = n->cfg.n_in;
    g.pin = n->pin;
    g.nout = n->cfg.n_out;
    g.pout = n->pout;
    g.B = n->B;
    g.M = n->M;
    g.W = n->maxw;
    g.nl = n->nl;
    g.pitch = std::max(std::max(n->pin, n->pout), n->maxw) + 8;
    g.mu_in = n->mu_in;
    g.sd_in = n->sd_in;
    g.mu_out = n->mu_out;
    g.sd_out = n->sd_out;
    g.wb = n->wb;
    g.wtb = n->wtb;
    g.wb_ms = n->WB;
    g.params = n->params;
    g.p_ms = n->P;
    for (int l = 0; l < n->nl; ++l) g.L[l] = n->L[l];
    g.dg = n->z;
    g.x0t = n->x0t;
    g.at = n->at;
    g.dzt = n->dztl;
    g.dz_w = dz_width(n);
    g.loss_part = n->loss_part;
    return g;
}

// a wave for each column tile of the widest layer, at least 4 and at most 16
template <bool TRAIN>
avh_status launch_rows(const avh_mlp* n, const RowsArgs& g) {
    const int tiles = std::max(n->maxw, n->pout) / 16;
    hipLaunchKernelGGL(mlp_rows_kernel<TRAIN>, dim3((g.rows + ROWS - 1) / ROWS, n->M),
                       dim3(64 * std::max(4, std::min(16, tiles))), 2 * sizeof(uint16_t) * ROWS * (size_t)g.pitch,
                       n->stream, g);
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

// Loss and gradients of the minibatch rows idx[member][row0 ...] of the device
// data, and with `adam` the update of every parameter, in two launches.
avh_status fused_step(avh_mlp* n, long long row0, long long idx_ms, const AdamArgs* adam) {
    RowsArgs g = rows_args(n);
    g.Y = n->dy;
    g.idx = n->idx + row0;
    g.idx_ms = idx_ms;
    g.rows = n->B;
    avh_status r = launch_rows<true>(n, g);
    if (r) return r;
    UpdateArgs u;
    std::memset(&u, 0, sizeof u);
    u.a = adam ? *adam : adam_args(n);
    u.grad = n->grad;
    u.x0t = n->x0t;
    u.at = n->at;
    u.dzt = n->dztl;
    u.pin = n->pin;
    u.W = n->maxw;
    u.B = n->B;
    u.M = n->M;
    u.nl = n->nl;
    u.dz_w = dz_width(n);
    u.nout = n->cfg.n_out;
    int first = 0, outs = 0;
    for (int l = 0; l < n->nl; ++l) {
        u.first[l] = first;
        first += ((n->L[l].nout / 16) * ((n->L[l].nin + 31) / 32) + 3) / 4;
        outs += n->L[l].nout;
    }
    u.first[n->nl] = first;
    u.loss_part = n->loss_part;
    u.nparts = n->B / ROWS;
    u.loss = n->loss;
    u.bias_blocks = (outs + 255) / 256;
    const dim3 grid(u.bias_blocks + first, n->M);
    if (adam) hipLaunchKernelGGL(mlp_update_kernel<true>, grid, dim3(256), 0, n->stream, u);
    else hipLaunchKernelGGL(mlp_update_kernel<false>, grid, dim3(256), 0, n->stream, u);
    AVH_HIP(hipGetLastError());
    return AVH_OK;
}

avh_status ensure_outbuf(avh_mlp* n, long long count) {
    if (count <= n->ocap) return AVH_OK;
    (void)hipFree(n->outbuf);
    n->outbuf = nullptr;
    n->ocap = 0;
    AVH_HIP(hipMalloc(&n->outbuf, sizeof(float) * count));
    n->ocap = count;
    return AVH_OK;
}

// `count` members' blocks from `src` (the first's) to the host in the
// caller's order: packed on the device, so that the copy needs no pass of the
// host over its values
avh_status read_packed(avh_mlp* n, const float* src, int count, float* host) {
    PackArgs a;
    std::memset(&a, 0, sizeof a);
    long long np = 0, most = 0;
    for (int l = 0; l < n->nl; ++l) {
        a.L[l] = n->L[l];
        a.fin[l] = l == 0 ? n->cfg.n_in : n->cfg.width;
        a.fout[l] = l == n->nl - 1 ? n->cfg.n_out : n->cfg.width;
        a.off[l] = np;
        const long long vals = (long long)a.fin[l] * a.fout[l] + a.fout[l];
        np += vals;
        most = std::max(most, vals);
    }
    avh_status r = ensure_outbuf(n, np * count);
    if (r) return r;
    a.src = src;
    a.dst = n->outbuf;
    a.src_ms = n->P;
    a.dst_ms = np;
    hipLaunchKernelGGL(mlp_pack_kernel, dim3((unsigned int)((most + 255) / 256), n->nl, count), dim3(256), 0,
                       n->stream, a);
    AVH_HIP(hipGetLastError());
    AVH_HIP(hipMemcpyAsync(host, n->outbuf, sizeof(float) * np * count, hipMemcpyDeviceToHost, n->stream));
    AVH_HIP(hipStreamSynchronize(n->stream));
    return AVH_OK;
}

// One member's parameters, copied as they are and packed by the host.  Less
// than the launch of a pack kernel and its wait below HOST_PACK_MAX values (us
// of get_params, on the device / here: 24 / 13 for 500 values, 30 / 20 for
// 49e3, 41 / 35 for 116e3, 60 / 67 for 229e3).
constexpr long long HOST_PACK_MAX = 1 << 17;
avh_status read_member(avh_mlp* n, int member, float* host) {
    std::unique_ptr<float[]> h(new (std::nothrow) float[(size_t)n->P]);
    if (!h) return fail(AVH_ENOMEM, "host allocation failed");
    AVH_HIP(hipStreamSynchronize(n->stream));
    AVH_HIP(hipMemcpy(h.get(), n->params + member * n->P, sizeof(float) * n->P, hipMemcpyDeviceToHost));
    for (int l = 0; l < n->nl; ++l) {
        const LayerDesc& L = n->L[l];
        const int fin = l == 0 ? n->cfg.n_in : n->cfg.width;
        const int fout = l == n->nl - 1 ? n->cfg.n_out : n->cfg.width;
        for (int o = 0; o < fout; ++o, host += fin)
            std::memcpy(host, h.get() + L.w_off + (long long)o * L.nin, sizeof(float) * fin);
        std::memcpy(host, h.get() + L.b_off, sizeof(float) * fout);
        host += fout;
    }
    return AVH_OK;
}

// Outputs of every member for the first `rows` device rows, in data units,
// slab by slab of at most PREDICT_SLAB rows (the outputs of a call then take
// at most 16 MiB a member at 64 outputs).
constexpr long long PREDICT_SLAB = 65536;
avh_status fused_predict(avh_mlp* n, long long rows, float* out) {
    const long long slab = std::min(rows, PREDICT_SLAB);
    const long long need = slab * n->M * n->cfg.n_out;
    avh_status r = ensure_outbuf(n, need);
    if (r) return r;
    for (long long c0 = 0; c0 < rows; c0 += slab) {
        RowsArgs g = rows_args(n);
        g.rows = (int)std::min(slab, rows - c0);
        g.X = n->dx + c0 * n->cfg.n_in;
        g.out = n->outbuf;
        if ((r = launch_rows<false>(n, g))) return r;
        const size_t part = sizeof(float) * (size_t)g.rows * n->cfg.n_out;
        if (g.rows == rows) {
            AVH_HIP(hipMemcpyAsync(out, n->outbuf, part * n->M, hipMemcpyDeviceToHost, n->stream));
        } else {
            for (int mem = 0; mem < n->M; ++mem)
                AVH_HIP(hipMemcpyAsync(out + ((size_t)mem * rows + c0) * n->cfg.n_out,
                                       n->outbuf + (size_t)mem * g.rows * n->cfg.n_out, part, hipMemcpyDeviceToHost,
                                       n->stream));
        }
        AVH_HIP(hipStreamSynchronize(n->stream));
    }
    return AVH_OK;
}

avh_status upload_data(avh_mlp* n, const float* X, const float* Y, long long rows) {
    avh_status r = ensure_data(n, rows);
    if (r) return r;
    AVH_HIP(hipMemcpyAsync(n->dx, X, sizeof(float) * rows * n->cfg.n_in, hipMemcpyHostToDevice, n->stream));
    if (Y) AVH_HIP(hipMemcpyAsync(n->dy, Y, sizeof(float) * rows * n->cfg.n_out, hipMemcpyHostToDevice, n->stream));
    return AVH_OK;
}

}  // namespace

extern "C" {

avh_status avh_mlp_create(avh_ctx* ctx, const avh_mlp_config* cfg, avh_mlp** out) {
    if (!ctx || !cfg || !out) return fail(AVH_EINVAL, "null argument");
    *out = nullptr;
    if (cfg->n_in < 1 || cfg->n_out < 1 || cfg->width < 16 || cfg->width % 16 || cfg->hidden < 1 ||
        cfg->hidden > MAX_LAYERS - 1 || cfg->members < 1 || cfg->members > 64 || cfg->batch < 16 ||
        cfg->batch % 16 || cfg->batch > 4096 || cfg->n_in > 4096 || cfg->n_out > 4096 || cfg->width > 4096)
        return fail(AVH_EINVAL,
                    "bad network shape (width and batch multiples of 16, 1..7 hidden layers, 1..64 members)");
    AVH_HIP(hipSetDevice(ctx->device));
    auto n = new (std::nothrow) avh_mlp;
    if (!n) return fail(AVH_ENOMEM, "host allocation failed");
    n->device = ctx->device;
    n->cfg = *cfg;
    n->nl = cfg->hidden + 1;
    n->pin = pad16(cfg->n_in);
    n->pout = pad16(cfg->n_out);
    n->B = cfg->batch;
    n->M = cfg->members;
    n->maxw = cfg->width;
    long long P = 0, WB = 0;
    for (int l = 0; l < n->nl; ++l) {
        LayerDesc& L = n->L[l];
        L.nin = l == 0 ? n->pin : cfg->width;
        L.nout = l == n->nl - 1 ? n->pout : cfg->width;
        L.w_off = P;
        P += (long long)L.nin * L.nout;
        L.b_off = P;
        P += L.nout;
        L.wb_off = WB;
        WB += (long long)L.nin * L.nout;
    }
    n->P = P;
    n->WB = WB;
    n->fused = std::max(std::max(n->pin, n->pout), n->maxw) <= FUSED_MAX_DIM;
    const long long M = n->M, B = n->B, W = cfg->width, H = cfg->hidden;
    const long long dzw = B * std::max<long long>(W, n->pout);
    bool ok = hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) == hipSuccess;
    if (!ok) n->stream = nullptr;
    auto alloc = [&](void** p, size_t bytes) { ok = ok && hipMalloc(p, bytes) == hipSuccess; };
    alloc((void**)&n->params, sizeof(float) * M * P);
    alloc((void**)&n->m, sizeof(float) * M * P);
    alloc((void**)&n->v, sizeof(float) * M * P);
    alloc((void**)&n->grad, sizeof(float) * M * P);
    alloc((void**)&n->wb, 2 * M * WB);
    alloc((void**)&n->wtb, 2 * M * WB);
    alloc((void**)&n->x0t, 2 * M * B * n->pin);
    alloc((void**)&n->z, sizeof(float) * H * M * B * W);
    alloc((void**)&n->at, 2 * H * M * B * W);
    alloc((void**)&n->mu_in, sizeof(float) * cfg->n_in);
    alloc((void**)&n->sd_in, sizeof(float) * cfg->n_in);
    alloc((void**)&n->mu_out, sizeof(float) * cfg->n_out);
    alloc((void**)&n->sd_out, sizeof(float) * cfg->n_out);
    alloc((void**)&n->loss, sizeof(float) * M);
    if (n->fused) {
        alloc((void**)&n->dztl, 2 * M * n->nl * dzw);
        alloc((void**)&n->loss_part, sizeof(float) * M * (B / ROWS));
    } else {
        alloc((void**)&n->x0, 2 * M * B * n->pin);
        alloc((void**)&n->a, 2 * H * M * B * W);
        alloc((void**)&n->yhat, sizeof(float) * M * B * n->pout);
        alloc((void**)&n->yn, sizeof(float) * M * B * n->pout);
        for (int i = 0; i < 2; ++i) {
            alloc((void**)&n->dz[i], 2 * M * dzw);
            alloc((void**)&n->dzt[i], 2 * M * dzw);
        }
    }
    if (!ok) {
        free_mlp(n);
        return fail(AVH_ENOMEM, "device allocation failed");
    }
    ok = hipMemset(n->m, 0, sizeof(float) * M * P) == hipSuccess &&
         hipMemset(n->v, 0, sizeof(float) * M * P) == hipSuccess &&
         hipMemset(n->grad, 0, sizeof(float) * M * P) == hipSuccess;
    std::vector<float> zeros(std::max(cfg->n_in, cfg->n_out), 0.f), ones(std::max(cfg->n_in, cfg->n_out), 1.f);
    ok = ok && hipMemcpy(n->mu_in, zeros.data(), sizeof(float) * cfg->n_in, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(n->sd_in, ones.data(), sizeof(float) * cfg->n_in, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(n->mu_out, zeros.data(), sizeof(float) * cfg->n_out, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(n->sd_out, ones.data(), sizeof(float) * cfg->n_out, hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        free_mlp(n);
        return fail(AVH_EHIP, "device initialisation failed");
    }
    // initial weights and biases ~ U(-1/sqrt(fan_in), 1/sqrt(fan_in)) from
    // std::mt19937_64(seed + member), padded entries zero
    std::vector<float> h((size_t)(M * P), 0.f);
    for (long long mem = 0; mem < M; ++mem) {
        std::mt19937_64 gen(cfg->seed + (uint64_t)mem);
        std::uniform_real_distribution<float> U(-1.f, 1.f);
        for (int l = 0; l < n->nl; ++l) {
            const LayerDesc& L = n->L[l];
            const int fin = l == 0 ? cfg->n_in : cfg->width;
            const int fout = l == n->nl - 1 ? cfg->n_out : cfg->width;
            const float bound = 1.f / std::sqrt((float)fin);
            for (int o = 0; o < fout; ++o)
                for (int k = 0; k < fin; ++k) h[mem * P + L.w_off + (long long)o * L.nin + k] = U(gen) * bound;
            for (int o = 0; o < fout; ++o) h[mem * P + L.b_off + o] = U(gen) * bound;
        }
    }
    if (hipMemcpy(n->params, h.data(), sizeof(float) * M * P, hipMemcpyHostToDevice) != hipSuccess) {
        free_mlp(n);
        return fail(AVH_EHIP, "device initialisation failed");
    }
    avh_status r = cast_weights(n);
    if (!r && hipStreamSynchronize(n->stream) != hipSuccess) r = fail(AVH_EHIP, "hipStreamSynchronize failed");
    if (r) {
        free_mlp(n);
        return r;
    }
    *out = n;
    return AVH_OK;
}

avh_status avh_mlp_destroy(avh_mlp* n) {
    free_mlp(n);
    return AVH_OK;
}

avh_status avh_mlp_num_params(avh_mlp* n, int64_t* count) {
    if (!n || !count) return fail(AVH_EINVAL, "null argument");
    int64_t c = 0;
    for (int l = 0; l < n->nl; ++l) {
        const int fin = l == 0 ? n->cfg.n_in : n->cfg.width;
        const int fout = l == n->nl - 1 ? n->cfg.n_out : n->cfg.width;
        c += (int64_t)fin * fout + fout;
    }
    *count = c;
    return AVH_OK;
}

avh_status avh_mlp_set_normalization(avh_mlp* n, const float* in_mean, const float* in_std, const float* out_mean,
                                     const float* out_std) {
    if (!n || !in_mean || !in_std || !out_mean || !out_std) return fail(AVH_EINVAL, "null argument");
    for (int i = 0; i < n->cfg.n_in; ++i)
        if (!(in_std[i] > 0)) return fail(AVH_EINVAL, "input scales must be positive");
    for (int i = 0; i < n->cfg.n_out; ++i)
        if (!(out_std[i] > 0)) return fail(AVH_EINVAL, "output scales must be positive");
    AVH_HIP(hipSetDevice(n->device));
    AVH_HIP(hipStreamSynchronize(n->stream));
    AVH_HIP(hipMemcpy(n->mu_in, in_mean, sizeof(float) * n->cfg.n_in, hipMemcpyHostToDevice));
    AVH_HIP(hipMemcpy(n->sd_in, in_std, sizeof(float) * n->cfg.n_in, hipMemcpyHostToDevice));
    AVH_HIP(hipMemcpy(n->mu_out, out_mean, sizeof(float) * n->cfg.n_out, hipMemcpyHostToDevice));
    AVH_HIP(hipMemcpy(n->sd_out, out_std, sizeof(float) * n->cfg.n_out, hipMemcpyHostToDevice));
    return AVH_OK;
}

// Unpadded parameter order per member: for each layer, W[out][in] row-major
// then b[out].
avh_status avh_mlp_get_params(avh_mlp* n, int member, float* out) {
    if (!n || !out || member < 0 || member >= n->M) return fail(AVH_EINVAL, "bad argument");
    AVH_HIP(hipSetDevice(n->device));
    if (n->P < HOST_PACK_MAX) return read_member(n, member, out);
    return read_packed(n, n->params + member * n->P, 1, out);
}

avh_status avh_mlp_set_params(avh_mlp* n, int member, const float* in) {
    if (!n || !in || member < 0 || member >= n->M) return fail(AVH_EINVAL, "bad argument");
    AVH_HIP(hipSetDevice(n->device));
    AVH_HIP(hipStreamSynchronize(n->stream));
    std::vector<float> h(n->P, 0.f);
    size_t o = 0;
    for (int l = 0; l < n->nl; ++l) {
        const LayerDesc& L = n->L[l];
        const int fin = l == 0 ? n->cfg.n_in : n->cfg.width;
        const int fout = l == n->nl - 1 ? n->cfg.n_out : n->cfg.width;
        for (int r = 0; r < fout; ++r)
            for (int k = 0; k < fin; ++k) h[L.w_off + (long long)r * L.nin + k] = in[o++];
        for (int r = 0; r < fout; ++r) h[L.b_off + r] = in[o++];
    }
    AVH_HIP(hipMemcpy(n->params + member * n->P, h.data(), sizeof(float) * n->P, hipMemcpyHostToDevice));
    avh_status r = cast_weights(n);
    if (r) return r;
    AVH_HIP(hipStreamSynchronize(n->stream));
    return AVH_OK;
}

// Loss and gradients of every member on the same `batch` rows (no update):
// grads[member][num_params] in the get_params order, loss[member].
avh_status avh_mlp_gradients(avh_mlp* n, const float* X, const float* Y, int64_t rows, float* grads, float* loss) {
    if (!n || !X || !Y || !grads || !loss) return fail(AVH_EINVAL, "null argument");
    if (rows != n->B) return fail(AVH_EINVAL, "rows must equal the minibatch size");
    AVH_HIP(hipSetDevice(n->device));
    avh_status r = upload_data(n, X, Y, rows);
    if (r) return r;
    if ((r = ensure_idx(n, rows))) return r;
    std::vector<int> id(rows);
    for (int i = 0; i < rows; ++i) id[i] = i;
    AVH_HIP(hipMemcpyAsync(n->idx, id.data(), sizeof(int) * rows, hipMemcpyHostToDevice, n->stream));
    AVH_HIP(hipMemsetAsync(n->loss, 0, sizeof(float) * n->M, n->stream));
    if (n->fused) {
        if ((r = fused_step(n, 0, 0, nullptr))) return r;
    } else {
        if ((r = gather(n, 0, 0, (int)rows, true))) return r;
        if ((r = forward(n))) return r;
        if ((r = backward(n))) return r;
    }
    AVH_HIP(hipMemcpyAsync(loss, n->loss, sizeof(float) * n->M, hipMemcpyDeviceToHost, n->stream));
    return read_packed(n, n->grad, n->M, grads);
}

// One Adam step of every member from the gradients of the last
// avh_mlp_gradients / training step (for step-by-step checks).
avh_status avh_mlp_adam_step(avh_mlp* n, float lr) {
    if (!n) return fail(AVH_EINVAL, "null argument");
    AVH_HIP(hipSetDevice(n->device));
    avh_status r = adam_step(n, lr);
    if (r) return r;
    AVH_HIP(hipStreamSynchronize(n->stream));
    return AVH_OK;
}

// Minibatch Adam over `epochs` passes of the rows; each member visits the
// rows in its own seeded order (Fisher-Yates from std::mt19937_64(seed +
// 1000003 * (epoch + 1) + member), epochs counted over every call on this
// network), floor(rows / batch) steps per epoch;
// learning rate lr * (final_lr_fraction + (1 - final_lr_fraction) * (1 +
// cos(pi * step / steps)) / 2).  epoch_loss[e][member] = mean minibatch loss.
avh_status avh_mlp_train(avh_mlp* n, const float* X, const float* Y, int64_t rows, int epochs, float lr,
                         float final_lr_fraction, float* epoch_loss) {
    if (!n || !X || !Y) return fail(AVH_EINVAL, "null argument");
    if (rows < n->B || epochs < 1) return fail(AVH_EINVAL, "need at least one minibatch and one epoch");
    if (rows > (1ll << 30)) return fail(AVH_EINVAL, "too many rows");
    AVH_HIP(hipSetDevice(n->device));
    avh_status r = upload_data(n, X, Y, rows);
    if (r) return r;
    if ((r = ensure_idx(n, rows * n->M))) return r;
    const long long steps_per_epoch = rows / n->B;
    const long long total = steps_per_epoch * epochs;
    std::vector<int> perm((size_t)(rows * n->M));
    std::vector<float> lh(n->M);
    long long k = 0;
    for (int e = 0; e < epochs; ++e) {
        for (int mem = 0; mem < n->M; ++mem) {
            std::mt19937_64 gen(n->cfg.seed + 1000003ull * (uint64_t)(n->epochs_done + e + 1) + (uint64_t)mem);
            int* p = perm.data() + (size_t)mem * rows;
            for (long long i = 0; i < rows; ++i) p[i] = (int)i;
            for (long long i = rows - 1; i > 0; --i) {
                const long long j = (long long)(gen() % (uint64_t)(i + 1));
                std::swap(p[i], p[j]);
            }
        }
        AVH_HIP(hipMemcpyAsync(n->idx, perm.data(), sizeof(int) * rows * n->M, hipMemcpyHostToDevice, n->stream));
        AVH_HIP(hipMemsetAsync(n->loss, 0, sizeof(float) * n->M, n->stream));
        for (long long s = 0; s < steps_per_epoch; ++s, ++k) {
            const double c = 0.5 * (1.0 + std::cos(3.14159265358979323846 * (double)k / (double)total));
            const float lr_k = lr * (final_lr_fraction + (1.f - final_lr_fraction) * (float)c);
            if (n->fused) {
                const AdamArgs a = next_adam(n, lr_k);
                if ((r = fused_step(n, s * n->B, rows, &a))) return r;
                continue;
            }
            if ((r = gather(n, s * n->B, rows, n->B, true))) return r;
            if ((r = forward(n))) return r;
            if ((r = backward(n))) return r;
            if ((r = adam_step(n, lr_k))) return r;
        }
        AVH_HIP(hipMemcpyAsync(lh.data(), n->loss, sizeof(float) * n->M, hipMemcpyDeviceToHost, n->stream));
        AVH_HIP(hipStreamSynchronize(n->stream));
        if (epoch_loss)
            for (int mem = 0; mem < n->M; ++mem) epoch_loss[(size_t)e * n->M + mem] = lh[mem] / (float)steps_per_epoch;
    }
    n->epochs_done += epochs;
    return AVH_OK;
}

avh_status avh_mlp_set_weight_decay(avh_mlp* n, float weight_decay) {
    if (!n) return fail(AVH_EINVAL, "null argument");
    if (!(weight_decay >= 0.f) || weight_decay > 1.f) return fail(AVH_EINVAL, "weight decay must be in [0, 1]");
    n->wd = weight_decay;
    return AVH_OK;
}

// Outputs of every member for `rows` inputs, in data units:
// out[member][row][n_out].
avh_status avh_mlp_predict(avh_mlp* n, const float* X, int64_t rows, float* out) {
    if (!n || !X || !out) return fail(AVH_EINVAL, "null argument");
    if (rows < 1 || rows > (1ll << 30)) return fail(AVH_EINVAL, "bad row count");
    AVH_HIP(hipSetDevice(n->device));
    avh_status r = upload_data(n, X, nullptr, rows);
    if (r) return r;
    if (n->fused) return fused_predict(n, rows, out);
    const long long padded = (rows + n->B - 1) / n->B * n->B;
    if ((r = ensure_idx(n, padded))) return r;
    std::vector<int> id(padded);
    for (long long i = 0; i < padded; ++i) id[i] = (int)std::min(i, (long long)rows - 1);
    AVH_HIP(hipMemcpyAsync(n->idx, id.data(), sizeof(int) * padded, hipMemcpyHostToDevice, n->stream));
    std::vector<float> mu(n->cfg.n_out), sd(n->cfg.n_out);
    AVH_HIP(hipMemcpyAsync(mu.data(), n->mu_out, sizeof(float) * n->cfg.n_out, hipMemcpyDeviceToHost, n->stream));
    AVH_HIP(hipMemcpyAsync(sd.data(), n->sd_out, sizeof(float) * n->cfg.n_out, hipMemcpyDeviceToHost, n->stream));
    std::vector<float> h((size_t)(n->M * n->B * n->pout));
    for (long long c0 = 0; c0 < rows; c0 += n->B) {
        const int cnt = (int)std::min<long long>(n->B, rows - c0);
        if ((r = gather(n, c0, 0, cnt, false))) return r;
        if ((r = forward(n))) return r;
        AVH_HIP(hipMemcpyAsync(h.data(), n->yhat, sizeof(float) * h.size(), hipMemcpyDeviceToHost, n->stream));
        AVH_HIP(hipStreamSynchronize(n->stream));
        for (int mem = 0; mem < n->M; ++mem)
            for (int i = 0; i < cnt; ++i)
                for (int o = 0; o < n->cfg.n_out; ++o)
                    out[((size_t)mem * rows + c0 + i) * n->cfg.n_out + o] =
                        h[((size_t)mem * n->B + i) * n->pout + o] * sd[o] + mu[o];
    }
    return AVH_OK;
}

}  // extern "C"
