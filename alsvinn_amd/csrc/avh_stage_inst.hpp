// Explicit instantiation of the stage launchers of one equation for every
// reconstruction, flux and grid dimension the equation supports.
#pragma once
#include "avh_batch.hpp"
#include "avh_line.hpp"
#include "avh_pair.hpp"
#include "avh_stage.hpp"
#include "avh_stage2d.hpp"
#include "avh_stage3d.hpp"

namespace avh {

// Host-side launcher types: one per (equation, reconstruction, flux, dim);
// `shape` selects one of the tile shapes below.
typedef hipError_t (*StageLauncher)(const StageParams& P, int shape, hipStream_t stream);
typedef hipError_t (*BatchLauncher)(const BatchParams& B, unsigned int nblocks, int shape, hipStream_t stream);
// Flux-only stage over a box of a reference Volume (P.n = box extent)
typedef hipError_t (*VolumeLauncher)(const StageParams& P, const VolumeParams& V, hipStream_t stream);

// Tile shapes the stage kernels are built for; the autotuner times them on
// the solver's own grid and keeps the fastest.  Every shape computes each
// interface flux and each cell update with the same operations in the same
// order, so the choice never changes a result bit.
//   1D (grids above avh_line.hpp's): (cells, threads) = (256, 256), with
//       RK3's last two stages in one launch, or (64, 64).
//   2D: a flux pass costs a wavefront its full instruction stream however few
//       of its lanes have an item, so the shapes' items sit just under their
//       threads.  32x15 on 256 threads (255 x / 256 y turns of two
//       interfaces) and 32x11 on 192 do the least work a cell and take the
//       large grids.  On smaller ones a workgroup's chain is what counts:
//       16x15 on 512 threads, 32x15 on 1024 and 16x7 on 256 evaluate both
//       directions side by side, one interface a thread (a lone tile takes
//       5.6, 7.7 and 4.8 us, 32x15 on 256 threads 8.9).  us of an RK3 stage
//       pair, 32x15 on 256 / 16x15 on 512 / 16x7: 64^2 17.9 / 11.2 / 9.6,
//       256^2 19.8 / 17.3 / 18.8, 501x333 27.4 / 25.9 / 33.8, 1024^2
//       91 / 112 / 165; 700x300, eno3, hll, first stage: 16.4, 32x15 on 1024
//       threads 15.5.
//   3D: 16x15, 17x14 or 14x17 columns marching through chunks of planes, 256
//       threads (at most 255 interfaces a plane in each direction: one turn;
//       the threads past the columns only work on the planes); the three
//       waste different parts of a grid that they do not divide (97x83x61:
//       42, 36 and 35 columns, 159 / 145 / 147 us of stages a step; 119x98x64
//       203 / 189 / 211, 128^3 447 / 482 / 473).  A chunk pays a z flux
//       and the loads of its window before its first plane, so the best length
//       is the one that fills the CUs evenly (march_chunk; the fixed lengths
//       stand beside it for grids where its model is off).  us of an RK3 stage
//       pair, 4 / 8 / 16 / 32 planes and march_chunk's: 200x150x120
//       566 / 539 / 582 / 700 / 528, 128^3 317 / 313 / 352 / 449 / 302, 64^3
//       76 / 87 / 159 / 299 / 64, 160^3 616 / 559 / 585 / 710 / 555.
// How often each is the fastest (a step's launches, seven schemes from none
// with forward euler to eno3 with rk3): in 2D on 18 grids from 32^2 to 2048^2,
// 17x3000 and 3000x9 among them, 32x15 on 256 44 times, 16x15 38, 16x7 26, 32x15
// on 1024 17 and 32x11 once, by 0.4 %; in 3D on 16 grids from 16^3 to 256^3,
// 300x200x5 and 64x64x400 among them, march_chunk's length in one of the three
// columns 79 times, 2 planes 12 (by 1.4 % at most), 4 planes 9 (8 %: 128^3, none,
// hll, forward euler 89 us against 97), 16 planes 9 (1.2 %) and 32 planes 3 (0.2 %).
constexpr int NSHAPES1 = 2, NSHAPES2 = 5, NSHAPES3 = 7;
constexpr int SHAPE1_TX[NSHAPES1] = {256, 64};
constexpr int SHAPE2_TX[NSHAPES2] = {32, 16, 16, 32, 32};
constexpr int SHAPE2_TY[NSHAPES2] = {11, 15, 7, 15, 15};
constexpr int SHAPE2_NT[NSHAPES2] = {192, 512, 256, 256, 1024};
constexpr int SHAPE3_TX[NSHAPES3] = {16, 16, 17, 14, 16, 16, 16};
constexpr int SHAPE3_TY[NSHAPES3] = {15, 15, 14, 17, 15, 15, 15};
constexpr int SHAPE3_LZ[NSHAPES3] = {4, 0, 0, 0, 16, 2, 32};  // 0: march_chunk

inline int num_shapes(int dim) { return dim == 1 ? NSHAPES1 : (dim == 2 ? NSHAPES2 : NSHAPES3); }

template <class EQ, int RECON, class FLUX, int DIM, int S>
struct KernelFor;
template <class EQ, int RECON, class FLUX, int S>
struct KernelFor<EQ, RECON, FLUX, 1, S> {
    typedef StageKernel1<EQ, RECON, FLUX, SHAPE1_TX[S], SHAPE1_TX[S]> type;
};
template <class EQ, int RECON, class FLUX, int S>
struct KernelFor<EQ, RECON, FLUX, 2, S> {
    typedef TileKernel2<EQ, RECON, FLUX, SHAPE2_TX[S], SHAPE2_TY[S], SHAPE2_NT[S]> type;
};
// 2D shapes whose RK stages are each compiled for their mode (the shapes
// the autotuner takes most); those kernels index cells with 32-bit values, so
// they serve grids of fewer than 2^29 cells (per sample in a batch)
constexpr bool SHAPE2_BY_MODE[NSHAPES2] = {false, true, true, true, true};
constexpr long long MODE_KERNEL_MAX_CELLS = 1ll << 29;
template <class EQ, int RECON, class FLUX, int S, int MODE>
struct KernelForMode {
    typedef TileKernel2<EQ, RECON, FLUX, SHAPE2_TX[S], SHAPE2_TY[S], SHAPE2_NT[S], MODE> type;
};

// stage tiles (workgroups) covering one grid of the 1D / 2D kernels
inline unsigned int stage_tiles(const int* n, int dim, int shape) {
    if (dim == 1) return (unsigned int)((n[0] + SHAPE1_TX[shape] - 1) / SHAPE1_TX[shape]);
    return (unsigned int)(((n[0] + SHAPE2_TX[shape] - 1) / SHAPE2_TX[shape]) *
                          ((n[1] + SHAPE2_TY[shape] - 1) / SHAPE2_TY[shape]));
}

template <class K>
hipError_t launch_batch_k(const BatchParams& B, unsigned int nblocks, hipStream_t stream) {
    hipLaunchKernelGGL(batch_stage_kernel<K>, dim3(nblocks), dim3(K::NTHREADS), 0, stream, B);
    return hipGetLastError();
}

template <class EQ, int RECON, class FLUX, int DIM>
hipError_t launch_batch_stage(const BatchParams& B, unsigned int nblocks, int shape, hipStream_t stream) {
    if constexpr (DIM == 3) {
        return hipErrorInvalidValue;
    } else if constexpr (DIM == 1) {
        switch (shape) {
        case 0: return launch_batch_k<typename KernelFor<EQ, RECON, FLUX, 1, 0>::type>(B, nblocks, stream);
        case 1: return launch_batch_k<typename KernelFor<EQ, RECON, FLUX, 1, 1>::type>(B, nblocks, stream);
        }
        return hipErrorInvalidValue;
    } else {
#define AVH_BATCH_MODES(S)                                                                                  \
    case S:                                                                                                 \
        if constexpr (SHAPE2_BY_MODE[S]) {                                                                  \
            if (!small) {                                                                                   \
            } else if (B.mode == MODE_L)                                                                    \
                return launch_batch_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_L>::type>(B, nblocks, \
                                                                                               stream);     \
            else if (B.mode == MODE_RK2_2)                                                                  \
                return launch_batch_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_RK2_2>::type>(        \
                    B, nblocks, stream);                                                                    \
            else if (B.mode == MODE_RK3_2)                                                                  \
                return launch_batch_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_RK3_2>::type>(        \
                    B, nblocks, stream);                                                                    \
            else if (B.mode == MODE_RK3_3)                                                                  \
                return launch_batch_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_RK3_3>::type>(        \
                    B, nblocks, stream);                                                                    \
        }                                                                                                   \
        return launch_batch_k<typename KernelFor<EQ, RECON, FLUX, 2, S>::type>(B, nblocks, stream);
        bool small = true;
        for (int i = 0; i < B.ngroups; ++i) small = small && B.g[i].ncells < MODE_KERNEL_MAX_CELLS;
        switch (shape) {
            AVH_BATCH_MODES(0)
            AVH_BATCH_MODES(1)
            AVH_BATCH_MODES(2)
            AVH_BATCH_MODES(3)
            AVH_BATCH_MODES(4)
        }
#undef AVH_BATCH_MODES
        return hipErrorInvalidValue;
    }
}

template <class K>
hipError_t launch_stage_k(const StageParams& P, hipStream_t stream) {
    hipLaunchKernelGGL(stage_kernel<K>, dim3(K::tiles(P.n)), dim3(K::NTHREADS), 0, stream, P);
    return hipGetLastError();
}

// Planes per chunk for a box of n cells, by a model of the launch.  The
// workgroups of a CU share its FP64 pipe, so a launch takes as long as the CU
// with the most of them, each worth its planes and about one more for its
// prologue; one alone leaves about a quarter of the pipe idle.
// 128^3, 16x15 columns, us of a volume substep's launch at 8 / 13 / 16 / 32
// planes and at the 19 this picks: 165 / 163 / 192 / 240 and 158.
// A chunk past the box is the box, so longer ones are not tried (each try costs
// a division, and a call over a small box is 31 us in all).
// `thin`: one plane where even that gives each CU no more than one workgroup,
// since what is left is a workgroup's chain.  us of a call of
// avh_numerical_flux on boxes of 128^3 (64^3), euler3 weno2, with chunks of two
// planes and more, and so: 2 cells in z 36.7 -> 33.0 (35.9 -> 31.5), in x
// 45.3 -> 45.3 (38.6 -> 34.1), in y 41.4 -> 41.3 (36.5 -> 33.7), a 2x2 pencil
// along x 35.8 -> 31.4, along z 36.6 -> 32.2, a 2x2x2 corner 35.1 -> 31.2; one
// workgroup per 8x4x4 brick takes 38.0 (32.7), 49.2 (38.5), 41.1 (35.4), 31.8,
// 39.1 and 31.7.  Not past one workgroup a CU: burgers eno2, 128x128x8 in 576
// workgroups of one plane 33.3, in 288 of two 31.1.
template <class K>
int march_chunk(const int* n, bool thin = false, long long* least = nullptr) {
    const unsigned int CUS = 256;
    const unsigned int columns = K::tiles(n, n[2]);
    const int longest = n[2] < 64 ? n[2] : 64;
    const bool single = longest == 1 || (thin && (long long)columns * n[2] <= CUS);
    int best = 0;
    long long cost = 0;
    for (int lz = single ? 1 : 2; lz <= (single ? 1 : longest); ++lz) {
        const long long per_cu = (columns * (unsigned int)((n[2] + lz - 1) / lz) + CUS - 1) / CUS;
        const long long c = (2 * per_cu < 3 ? 3 : 2 * per_cu) * (lz + 1);
        if (!best || c < cost) {
            best = lz;
            cost = c;
        }
    }
    if (least) *least = cost;
    return best;
}

template <class K>
hipError_t launch_march_k(const StageParams& P, hipStream_t stream) {
    hipLaunchKernelGGL(march_kernel3<K>, dim3(K::tiles(P.n, P.lz)), dim3(K::NT), 0, stream, P);
    return hipGetLastError();
}

// one column tile: each stage mode has a kernel compiled for it; flux-only
// launches, and grids whose cells need 64-bit indices, take the kernel that
// reads the mode
template <class EQ, int RECON, class FLUX, int TX, int TY>
hipError_t launch_march(StageParams P, int lz, hipStream_t stream) {
    P.lz = lz ? lz : march_chunk<MarchKernel3<EQ, RECON, FLUX, TX, TY, 256>>(P.n);
    if (P.ncells < MODE_KERNEL_MAX_CELLS) {
        switch (P.mode) {
        case MODE_L: return launch_march_k<MarchKernel3<EQ, RECON, FLUX, TX, TY, 256, MODE_L>>(P, stream);
        case MODE_RK2_2: return launch_march_k<MarchKernel3<EQ, RECON, FLUX, TX, TY, 256, MODE_RK2_2>>(P, stream);
        case MODE_RK3_2: return launch_march_k<MarchKernel3<EQ, RECON, FLUX, TX, TY, 256, MODE_RK3_2>>(P, stream);
        case MODE_RK3_3: return launch_march_k<MarchKernel3<EQ, RECON, FLUX, TX, TY, 256, MODE_RK3_3>>(P, stream);
        }
    }
    return launch_march_k<MarchKernel3<EQ, RECON, FLUX, TX, TY, 256>>(P, stream);
}

template <class EQ, int RECON, class FLUX, int DIM>
hipError_t launch_stage(const StageParams& P, int shape, hipStream_t stream) {
    if constexpr (DIM == 3) {
        if (shape < 0 || shape >= NSHAPES3) return hipErrorInvalidValue;
        switch (SHAPE3_TX[shape]) {
        case 14: return launch_march<EQ, RECON, FLUX, 14, 17>(P, SHAPE3_LZ[shape], stream);
        case 17: return launch_march<EQ, RECON, FLUX, 17, 14>(P, SHAPE3_LZ[shape], stream);
        }
        return launch_march<EQ, RECON, FLUX, 16, 15>(P, SHAPE3_LZ[shape], stream);
    } else if constexpr (DIM == 1) {
        switch (shape) {
        case 0: return launch_stage_k<typename KernelFor<EQ, RECON, FLUX, 1, 0>::type>(P, stream);
        case 1: return launch_stage_k<typename KernelFor<EQ, RECON, FLUX, 1, 1>::type>(P, stream);
        }
        return hipErrorInvalidValue;
    } else {
#define AVH_STAGE_MODES(S)                                                                                  \
    case S:                                                                                                 \
        if constexpr (SHAPE2_BY_MODE[S]) {                                                                  \
            if (P.ncells >= MODE_KERNEL_MAX_CELLS) {                                                        \
            } else if (P.mode == MODE_L)                                                                    \
                return launch_stage_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_L>::type>(P, stream); \
            else if (P.mode == MODE_RK2_2)                                                                  \
                return launch_stage_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_RK2_2>::type>(P,      \
                                                                                                 stream);   \
            else if (P.mode == MODE_RK3_2)                                                                  \
                return launch_stage_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_RK3_2>::type>(P,      \
                                                                                                 stream);   \
            else if (P.mode == MODE_RK3_3)                                                                  \
                return launch_stage_k<typename KernelForMode<EQ, RECON, FLUX, S, MODE_RK3_3>::type>(P,      \
                                                                                                 stream);   \
        }                                                                                                   \
        return launch_stage_k<typename KernelFor<EQ, RECON, FLUX, 2, S>::type>(P, stream);
        switch (shape) {
            AVH_STAGE_MODES(0)
            AVH_STAGE_MODES(1)
            AVH_STAGE_MODES(2)
            AVH_STAGE_MODES(3)
            AVH_STAGE_MODES(4)
        }
#undef AVH_STAGE_MODES
        return hipErrorInvalidValue;
    }
}

// The reference-Volume kernels: 1D 256 cells, 2D 32x15 or 16x7, 3D columns.  P.mode is MODE_FLUX_ONLY, or MODE_RK3_3 for the
// combination V describes.
// 2D boxes of few 16x7 tiles take these: a workgroup's chain is then all there
// is, and 32x15's threads march along two interfaces.  us of a call of
// avh_numerical_flux, weno2 hll3, one interface at a time in 32x15 tiles, 32x15
// so and 16x7: a strip of 2x200 cells 41.6 / 38.7 / 27.9, of 200x2 30.7 / 31.2 /
// 27.2, 128^2 (152 tiles) 33.1 / 31.8 / 28.9, 200x150 (286) 33.4 / 31.8 / 30.3,
// 200^2 (377) 33.6 / 32.1 / 31.4, 200x300 (559) 34.3 / 32.6 / 33.7.
constexpr unsigned int VOLUME2_SMALL_TILES = 384;
template <class EQ, int RECON, class FLUX>
struct VolumeKernel1 {
    typedef StageKernel1<EQ, RECON, FLUX, 256, 256> type;
};
template <class EQ, int RECON, class FLUX>
struct VolumeKernel2 {
    typedef TileKernel2<EQ, RECON, FLUX, 32, 15, 256> type;
    typedef TileKernel2<EQ, RECON, FLUX, 16, 7, 256> small;  // both directions at once, one interface a thread
};

template <class K>
hipError_t launch_volume_k(const StageParams& P, const VolumeParams& V, hipStream_t stream) {
    hipLaunchKernelGGL(volume_stage_kernel<K>, dim3(K::tiles(P.n)), dim3(K::NTHREADS), 0, stream, P, V);
    return hipGetLastError();
}

template <class K>
hipError_t launch_volume_march_k(const StageParams& P, const VolumeParams& V, int lz, hipStream_t stream) {
    StageParams Q = P;
    Q.lz = lz;
    hipLaunchKernelGGL(volume_march_kernel3<K>, dim3(K::tiles(P.n, lz)), dim3(K::NT), 0, stream, Q, V);
    return hipGetLastError();
}

// Boxes at most NARROW_TX cells wide in x (a strip or a pencil beside a
// neighbour): in 4x24 columns on 128 threads.  In 16x15 ones most lanes idle,
// and the fifteen rows that a workgroup then loads, a cache line each and all at
// once, are what it waits for.  As few planes as leave at most four workgroups a
// CU, which is all of them at once.  us of a call of avh_numerical_flux, euler3
// hll3, none / weno2 / eno3, one workgroup per 8x4x4 brick, in 16x15 columns and
// so: a pencil along y of 128^3 31.0 / 36.0 / 33.5, 35.5 / 38.6 / 34.7 and
// 30.7 / 31.2 / 32.6; a strip in x of 4x100x100 39.9 / 43.5 / - , 42.2 / 46.0 / -
// and 35.0 / 36.9 / - , of 128^3 45.4 / 48.6 / 59.0, 41.3 / 45.2 / 47.6 and
// 38.6 / 40.7 / 43.0, of 200x300x100 62.8 / 70.6 / 87.9, 51.7 / 59.2 / 63.6 and
// 41.5 / 47.3 / 50.6.  Pencils along z lose past some 500 cells (2x2x900 34.9 /
// 37.8 / 39.7, 38.7 / 41.0 / 43.0 and 40.3 / 42.0 / 43.9): a workgroup a plane, and
// each reports its wave speeds.
constexpr int NARROW_TX = 4;
template <class K>
int narrow_chunk(const int* n) {
    const unsigned int most = 4 * 256;
    const unsigned int columns = K::tiles(n, n[2]);
    const unsigned int chunks = most / columns;  // along z
    return chunks < 2 ? n[2] : (int)((n[2] + chunks - 1) / chunks);
}

// The columns whose launch the model finds shortest (a volume has no
// autotuner): their workgroups do the same work a plane, so the costs compare.
// us of an RK3 step through the volume interfaces, 16x15 alone and so: 97x83x61
// 289 and 273, 119x98x64 340 and 327, 33x110x50 216 and 200, 128^3 the same.
template <class EQ, int RECON, class FLUX, int MODE>
hipError_t launch_volume_march(const StageParams& P, const VolumeParams& V, hipStream_t stream) {
    typedef MarchKernel3<EQ, RECON, FLUX, 16, 15, 256, MODE, true> A;
    typedef MarchKernel3<EQ, RECON, FLUX, 17, 14, 256, MODE, true> B;
    typedef MarchKernel3<EQ, RECON, FLUX, 14, 17, 256, MODE, true> C;
    typedef MarchKernel3<EQ, RECON, FLUX, NARROW_TX, 24, 128, MODE, true> D;
    if (P.n[0] <= NARROW_TX) return launch_volume_march_k<D>(P, V, narrow_chunk<D>(P.n), stream);
    long long a, b, c;
    const int la = march_chunk<A>(P.n, true, &a), lb = march_chunk<B>(P.n, true, &b), lc = march_chunk<C>(P.n, true, &c);
    if (a <= b && a <= c) return launch_volume_march_k<A>(P, V, la, stream);
    return b <= c ? launch_volume_march_k<B>(P, V, lb, stream) : launch_volume_march_k<C>(P, V, lc, stream);
}

template <class EQ, int RECON, class FLUX, int DIM>
hipError_t launch_volume_stage(const StageParams& P, const VolumeParams& V, hipStream_t stream) {
    if constexpr (DIM == 3) {
        if (P.mode == MODE_FLUX_ONLY)
            return launch_volume_march<EQ, RECON, FLUX, MODE_FLUX_ONLY>(P, V, stream);
        return launch_volume_march<EQ, RECON, FLUX, MODE_RK3_3>(P, V, stream);
    } else {
        typedef typename std::conditional<DIM == 1, VolumeKernel1<EQ, RECON, FLUX>,
                                          VolumeKernel2<EQ, RECON, FLUX>>::type Kernels;
        if constexpr (DIM == 2) {
            typedef typename Kernels::small S;
            if (S::tiles(P.n) <= VOLUME2_SMALL_TILES) return launch_volume_k<S>(P, V, stream);
        }
        return launch_volume_k<typename Kernels::type>(P, V, stream);
    }
}

// Steps of a small 1D grid in one workgroup (avh_line.hpp), for burgers and
// euler1.
typedef hipError_t (*LineLauncher)(const LineParams& P, hipStream_t stream);

template <class K>
hipError_t launch_line_k(const LineParams& P, int threads, hipStream_t stream) {
    hipLaunchKernelGGL(line_kernel<K>, dim3(1), dim3(threads), K::lds_bytes(P.n), stream, P);
    return hipGetLastError();
}

template <class EQ, int RECON, class FLUX>
hipError_t launch_line(const LineParams& P, hipStream_t stream) {
    const int ni = P.bc == BC_PERIODIC ? P.n : P.n + 1;
    const int cpt = ni <= 512 ? 1 : (ni <= 1024 ? 2 : 4);
    const int threads = ((ni + cpt - 1) / cpt + 63) / 64 * 64;
    if (ni > line_interfaces(EQ::NV)) return hipErrorInvalidValue;
    if (cpt == 1) return launch_line_k<LineKernel<EQ, RECON, FLUX, 1>>(P, threads, stream);
    if (cpt == 2) return launch_line_k<LineKernel<EQ, RECON, FLUX, 2>>(P, threads, stream);
    if constexpr (EQ::NV == 1) return launch_line_k<LineKernel<EQ, RECON, FLUX, 4>>(P, threads, stream);
    return hipErrorInvalidValue;
}

// RK3's last two stages in one launch (avh_pair.hpp): shape 2 of 2D grids
// and shape 0 of 1D ones, where the grid is wide enough.
typedef hipError_t (*PairLauncher)(const StageParams& P, int shape, hipStream_t stream);  // as StageLauncher

template <class K>
hipError_t launch_pair_k(const StageParams& P, hipStream_t stream) {
    hipLaunchKernelGGL(pair_kernel<K>, dim3(K::tiles(P.n)), dim3(K::NTHREADS), 0, stream, P);
    return hipGetLastError();
}

template <class EQ, int RECON, class FLUX, int DIM>
hipError_t launch_pair(const StageParams& P, int, hipStream_t stream) {
    if constexpr (DIM == 1) return launch_pair_k<PairKernel<EQ, RECON, FLUX, 1, 240, 1, 256>>(P, stream);
    else return launch_pair_k<PairKernel<EQ, RECON, FLUX, 2, 16, 7, 512>>(P, stream);
}

// whether a shape's RK3 steps run their last two stages in one launch
inline bool pair_shape(int dim, int shape, const int* n, int ghosts) {
    if (dim > 2 || shape != (dim == 1 ? 0 : 2)) return false;
    for (int d = 0; d < dim; ++d)
        if (n[d] < 2 * ghosts) return false;
    return true;
}

struct Launchers {
    StageLauncher stage = nullptr;
    PairLauncher pair = nullptr;
    LineLauncher line = nullptr;
    BatchLauncher batch = nullptr;
    VolumeLauncher volume = nullptr;
};

template <class EQ, int RECON, class FLUX, int DIM>
Launchers launchers_of() {
    Launchers L;
    L.stage = &launch_stage<EQ, RECON, FLUX, DIM>;
    if (DIM < 3) L.batch = &launch_batch_stage<EQ, RECON, FLUX, DIM>;
    if constexpr (DIM < 3) L.pair = &launch_pair<EQ, RECON, FLUX, DIM>;
    if constexpr (DIM == 1 && EQ::NV <= 3) L.line = &launch_line<EQ, RECON, FLUX>;
    L.volume = &launch_volume_stage<EQ, RECON, FLUX, DIM>;
    return L;
}

template <class EQ, class FLUX, int DIM>
Launchers pick_recon(int recon) {
    switch (recon) {
    case RECON_NONE: return launchers_of<EQ, RECON_NONE, typename FLUX::template For<RECON_NONE>, DIM>();
    case RECON_WENO2: return launchers_of<EQ, RECON_WENO2, typename FLUX::template For<RECON_WENO2>, DIM>();
    case RECON_ENO2: return launchers_of<EQ, RECON_ENO2, typename FLUX::template For<RECON_ENO2>, DIM>();
    case RECON_ENO3: return launchers_of<EQ, RECON_ENO3, typename FLUX::template For<RECON_ENO3>, DIM>();
    }
    return Launchers();
}

// grids of one or two active axes, and of three where the caller's
// translation unit holds those kernels too
template <class EQ, class FLUX, int MAX_DIM = 3>
Launchers pick_dim(int recon, int dim) {
    if (dim == 1) return pick_recon<EQ, FLUX, 1>(recon);
    if constexpr (EQ::NSD >= 2) {
        if (dim == 2) return pick_recon<EQ, FLUX, 2>(recon);
    }
    if constexpr (EQ::NSD >= 3 && MAX_DIM >= 3) {
        if (dim == 3) return pick_recon<EQ, FLUX, 3>(recon);
    }
    return Launchers();
}

// flux ids follow avh_config: 0 godunov, 1 hll, 2 hll3
Launchers get_launchers_burgers(int recon, int flux, int dim);
Launchers get_launchers_euler1(int recon, int flux, int dim);
Launchers get_launchers_euler2(int recon, int flux, int dim);
Launchers get_launchers_euler3(int recon, int flux, int dim);
// euler3 on three active axes, one translation unit per reconstruction (they
// take most of the build's time)
Launchers get_launchers_euler3_3d_none(int flux);
Launchers get_launchers_euler3_3d_weno2(int flux);
Launchers get_launchers_euler3_3d_eno2(int flux);
Launchers get_launchers_euler3_3d_eno3(int flux);

}  // namespace avh
