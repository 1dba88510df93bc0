// GEMM update of the recursive triangular solve / multiply on gfx950 MFMA.
//
//   C = beta*C + alpha*op(X)*op(Y)      op(X): M x K, op(Y): K x N, C: M x N
//
// Replaces matmul! (src/matmul.jl:5-66) as used by GEMM_ADD!/GEMM_SUB!
// (src/matmul.jl:69-80) from unified_rec (src/rectrxm.jl:164-192).  The
// reference kernel computes one output per work-item from 32x32 LDS tiles;
// here every wave owns a (BM/WM) x (BN/WN) block of C held in MFMA
// accumulators, operands are staged through double-buffered LDS, and the
// alpha pre/post scaling of unified_rectrxm! (src/rectrxm.jl:64,72) is folded
// into beta/alpha so B is never swept separately.
#include "nla_gemm_tile.h"
#include "nla_internal.h"

namespace nla {

// TRI: triangle mask on one operand (see GemmArgs::tri).  C is not declared
// __restrict__: a leaf update writes the strip it reads.
template <typename T, int BM, int BN, int BK, int WM, int WN, bool TX, bool TY, int TRI>
__global__ __launch_bounds__(WM *WN * 64) void gemm_kernel(int64_t M, int64_t N, int64_t K, T alpha,
                                                           const T *__restrict__ X, int64_t ldx,
                                                           const T *__restrict__ Y, int64_t ldy, T beta,
                                                           T *C, int64_t ldc, int tiles_m) {
    typedef TileLds<T, BM, BN, BK, WM, WN, TX, TY> L;
    __shared__ __attribute__((aligned(16))) T lds_x[L::X];
    __shared__ __attribute__((aligned(16))) T lds_y[L::Y];
    int tm, tn;
    tile_coords(gridDim.x, blockIdx.x, tiles_m, tm, tn);
    const int64_t row0 = (int64_t)tm * BM, col0 = (int64_t)tn * BN;
    const bool interior = row0 + BM <= M && col0 + BN <= N;
    if (interior)
        gemm_tile<T, BM, BN, BK, WM, WN, TX, TY, TRI, false>(M, N, K, alpha, X, ldx, Y, ldy, beta, C, ldc,
                                                                 row0, col0, (NLA_LDS T *)lds_x,
                                                                 (NLA_LDS T *)lds_y);
    else
        gemm_tile<T, BM, BN, BK, WM, WN, TX, TY, TRI, true>(M, N, K, alpha, X, ldx, Y, ldy, beta, C, ldc,
                                                                row0, col0, (NLA_LDS T *)lds_x,
                                                                (NLA_LDS T *)lds_y);
}

// A triangular operand gives the tiles k-ranges from one k-step to all of K.
// With one work-group per tile, the work-groups that draw the long tiles set
// the runtime (the hardware hands a CU its next work-group in a fixed
// rotation, so a CU keeps meeting tiles of the same rows).  Here a grid of
// resident work-groups takes tiles from a counter instead, longest first;
// all columns (rows) of a row (column) of tiles are taken together, so the
// work-groups running at one time share that operand panel in L2.  *queue
// must be zero at launch; every work-group leaves once the counter passes
// the tile count.
template <typename T, int BM, int BN, int BK, int WM, int WN, bool TX, bool TY, int TRI>
__global__ __launch_bounds__(WM *WN * 64) void gemm_tri_queue_kernel(int64_t M, int64_t N, int64_t K, T alpha,
                                                                     const T *__restrict__ X, int64_t ldx,
                                                                     const T *__restrict__ Y, int64_t ldy, T beta,
                                                                     T *C, int64_t ldc, int tiles_m, int tiles_n,
                                                                     int *queue) {
    static_assert(TRI >= 1 && TRI <= 4, "triangular operand expected");
    typedef TileLds<T, BM, BN, BK, WM, WN, TX, TY> L;
    __shared__ __attribute__((aligned(16))) T lds_x[L::X];
    __shared__ __attribute__((aligned(16))) T lds_y[L::Y];
    __shared__ int s_tile;
    const int ntiles = tiles_m * tiles_n;
    for (;;) {
        if (threadIdx.x == 0) s_tile = atomicAdd(queue, 1);
        __syncthreads();
        const int t = s_tile;
        __syncthreads();  // read by all before thread 0 takes the next one
        if (t >= ntiles) break;
        int tm, tn;
        if (TRI == 1) {  // k-range grows with the row: last rows first
            tm = tiles_m - 1 - t / tiles_n;
            tn = t % tiles_n;
        } else if (TRI == 2) {
            tm = t / tiles_n;
            tn = t % tiles_n;
        } else if (TRI == 3) {
            tn = t / tiles_m;
            tm = t % tiles_m;
        } else {
            tn = tiles_n - 1 - t / tiles_m;
            tm = t % tiles_m;
        }
        const int64_t row0 = (int64_t)tm * BM, col0 = (int64_t)tn * BN;
        const bool interior = row0 + BM <= M && col0 + BN <= N;
        if (interior)
            gemm_tile<T, BM, BN, BK, WM, WN, TX, TY, TRI, false>(M, N, K, alpha, X, ldx, Y, ldy, beta, C, ldc,
                                                                     row0, col0, (NLA_LDS T *)lds_x,
                                                                     (NLA_LDS T *)lds_y);
        else
            gemm_tile<T, BM, BN, BK, WM, WN, TX, TY, TRI, true>(M, N, K, alpha, X, ldx, Y, ldy, beta, C, ldc,
                                                                    row0, col0, (NLA_LDS T *)lds_x,
                                                                    (NLA_LDS T *)lds_y);
    }
}

template <typename T, int BM, int BN, int BK, int WM, int WN, bool TX, bool TY, int TRI>
static hipError_t launch_cfg(const GemmArgs<T> &a, hipStream_t s) {
    int tiles_m = (int)((a.M + BM - 1) / BM);
    int tiles_n = (int)((a.N + BN - 1) / BN);
    int G = tiles_m * tiles_n;
    if constexpr (TRI != 0) {
        if (a.queue != nullptr && a.leaf == 0) {
            constexpr int NT = WM * WN * 64;
            static const int occ = [] {
                int o = 0;
                if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                        &o, (const void *)gemm_tri_queue_kernel<T, BM, BN, BK, WM, WN, TX, TY, TRI>, NT, 0) !=
                    hipSuccess)
                    o = 1;
                return o > 0 ? o : 1;
            }();
            int dev = 0, cus = 0;
            hipError_t e = hipGetDevice(&dev);
            if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
            if (e != hipSuccess) return e;
            int grid = cus * occ < G ? cus * occ : G;
            hipLaunchKernelGGL((gemm_tri_queue_kernel<T, BM, BN, BK, WM, WN, TX, TY, TRI>), dim3(grid), dim3(NT),
                               0, s, a.M, a.N, a.K, a.alpha, a.X, a.ldx, a.Y, a.ldy, a.beta, a.C, a.ldc, tiles_m,
                               tiles_n, a.queue);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, BK, WM, WN, TX, TY, TRI>), dim3(G), dim3(WM * WN * 64), 0, s, a.M,
                       a.N, a.K, a.alpha, a.X, a.ldx, a.Y, a.ldy, a.beta, a.C, a.ldc, tiles_m);
    return hipGetLastError();
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int TRI>
static hipError_t launch_trans(const GemmArgs<T> &a, hipStream_t s) {
    if (!a.tx && !a.ty) return launch_cfg<T, BM, BN, BK, WM, WN, false, false, TRI>(a, s);
    if (a.tx && !a.ty) return launch_cfg<T, BM, BN, BK, WM, WN, true, false, TRI>(a, s);
    if (!a.tx && a.ty) return launch_cfg<T, BM, BN, BK, WM, WN, false, true, TRI>(a, s);
    return launch_cfg<T, BM, BN, BK, WM, WN, true, true, TRI>(a, s);
}

template <typename T, int BM, int BN, int BK, int WM, int WN>
static hipError_t launch_tri(const GemmArgs<T> &a, hipStream_t s) {
    switch (a.tri) {
        case 1: return launch_trans<T, BM, BN, BK, WM, WN, 1>(a, s);
        case 2: return launch_trans<T, BM, BN, BK, WM, WN, 2>(a, s);
        case 3: return launch_trans<T, BM, BN, BK, WM, WN, 3>(a, s);
        case 4: return launch_trans<T, BM, BN, BK, WM, WN, 4>(a, s);
        default: return launch_trans<T, BM, BN, BK, WM, WN, 0>(a, s);
    }
}

// A dense product with one triangular operand: op(X) (TRI 1/2, op(Y) dense,
// untransposed) or op(Y) (TRI 3/4, op(X) dense, untransposed) -- the shapes
// of the residual alpha*B - op(A)*X and alpha*B - X*op(A).
template <typename T, int BM, int BN, int BK, int WM, int WN>
static hipError_t launch_tri_dense(const GemmArgs<T> &a, hipStream_t s) {
    switch (a.tri) {
        case 1:
            if (a.ty) return hipErrorInvalidValue;
            return a.tx ? launch_cfg<T, BM, BN, BK, WM, WN, true, false, 1>(a, s)
                        : launch_cfg<T, BM, BN, BK, WM, WN, false, false, 1>(a, s);
        case 2:
            if (a.ty) return hipErrorInvalidValue;
            return a.tx ? launch_cfg<T, BM, BN, BK, WM, WN, true, false, 2>(a, s)
                        : launch_cfg<T, BM, BN, BK, WM, WN, false, false, 2>(a, s);
        case 3:
            if (a.tx) return hipErrorInvalidValue;
            return a.ty ? launch_cfg<T, BM, BN, BK, WM, WN, false, true, 3>(a, s)
                        : launch_cfg<T, BM, BN, BK, WM, WN, false, false, 3>(a, s);
        case 4:
            if (a.tx) return hipErrorInvalidValue;
            return a.ty ? launch_cfg<T, BM, BN, BK, WM, WN, false, true, 4>(a, s)
                        : launch_cfg<T, BM, BN, BK, WM, WN, false, false, 4>(a, s);
        default:
            return launch_trans<T, BM, BN, BK, WM, WN, 0>(a, s);
    }
}

// Tile shape by the time its rounds take: ceil(tiles / CUs) rounds of the
// tile's area at the rate its shape reaches with full rounds, for K and
// the depth k0 that a round's start and end are worth.  Rates measured on
// MI355X (TFLOP/s): FP64 256 x 128 67, 128 x 128 62, 64 x 128 50; FP32
// 256 x 256 137 (one group per CU, so nothing hides its start and end),
// 128 x 128 131 (114 with ragged edges or one group per CU), 64 x 64 126.
// E.g. FP64 3000^3 1515 / 1230 / 1353 us, 6000 x 1024 x 1024
// 269 / 289 / 317; FP32 6000 x 2048 x 2048 550 / 446 / 415,
// 1024 x 8192 x 1024 256 / 140 / 144, 512 x 8192 x 512 - / 47 / 42,
// 3333 x 4444 x 555 186 / 170 / 162.
template <typename T>
int gemm_tile_shape(int64_t M, int64_t N, int64_t K, double *us) {
    auto cost = [&](int bm, int bn, double rate, int k0) {
        const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        return (double)((tiles + 255) / 256) * bm * bn / rate * (double)(K + k0);
    };
    double c[3];
    if constexpr (sizeof(T) == 8) {
        c[0] = cost(256, 128, 67, 0);
        c[1] = cost(128, 128, 62, 0);
        c[2] = cost(64, 128, 50, 0);
    } else {
        const bool slow = M % 128 != 0 || N % 128 != 0 || (M / 128) * (N / 128) <= 256;
        c[0] = cost(256, 256, 137, 100);
        c[1] = cost(128, 128, slow ? 114 : 131, 30);
        c[2] = cost(64, 64, 126, 30);
    }
    const int shape = c[0] <= c[1] && c[0] <= c[2] ? 0 : (c[1] <= c[2] ? 1 : 2);
    if (us != nullptr) *us = c[shape] * (2 * 256 * 1e-6);  // 2 flops on each of 256 CUs, TFLOP/s
    return shape;
}
template int gemm_tile_shape<float>(int64_t, int64_t, int64_t, double *);
template int gemm_tile_shape<double>(int64_t, int64_t, int64_t, double *);

template <typename T>
hipError_t launch_gemm_tiled(const GemmArgs<T> &a, hipStream_t s) {
    if (a.M <= 0 || a.N <= 0) return hipSuccess;
    if (a.leaf) {
        // one leaf (<= 64) along M (left) or N (right) and along K: a single
        // tile covers the leaf dimension, K is consumed in two steps.
        if (a.leaf == 1) {  // left: C (nb x m) = W (nb x nb) * B (nb x m)
            if (a.M > 64 || a.K > 64) return hipErrorInvalidValue;
            if constexpr (sizeof(T) == 8) return launch_tri<T, 64, 32, 32, 2, 2>(a, s);
            else return launch_tri<T, 64, 64, 32, 2, 2>(a, s);
        }
        // right: C (m x nb) = B (m x nb) * W (nb x nb)
        if (a.N > 64 || a.K > 64) return hipErrorInvalidValue;
        if constexpr (sizeof(T) == 8) return launch_tri<T, 32, 64, 32, 2, 2>(a, s);
        else return launch_tri<T, 64, 64, 32, 2, 2>(a, s);
    }
    const int shape = gemm_tile_shape<T>(a.M, a.N, a.K, nullptr);
    if constexpr (sizeof(T) == 8) {
        if (shape == 0) return launch_tri_dense<T, 256, 128, 16, 4, 2>(a, s);
        if (shape == 1) return launch_tri_dense<T, 128, 128, 16, 4, 2>(a, s);
        return launch_tri_dense<T, 64, 128, 16, 2, 2>(a, s);
    } else {
        if (a.tri) return hipErrorInvalidValue;  // triangular products are FP64 only
        if (shape == 0) return launch_trans<T, 256, 256, 32, 4, 4, 0>(a, s);
        if (shape == 1) return launch_trans<T, 128, 128, 32, 2, 2, 0>(a, s);
        return launch_trans<T, 64, 64, 32, 2, 2, 0>(a, s);
    }
}

// ---- grouped GEMM of the staged batched solver ----------------------------

// Work-groups take (gemm, tile) tasks from a counter until it passes ntasks;
// each task is one tile of one GEMM of the group, run by the same tile
// routine as the single GEMM.
template <typename T, int BM, int BN, int BK, int WM, int WN, bool TX, bool TY>
__global__ __launch_bounds__(WM *WN * 64) void grouped_gemm_kernel(const GroupGemm<T> *__restrict__ g,
                                                                   const int2 *__restrict__ tasks, int ntasks,
                                                                   int *counter) {
    typedef TileLds<T, BM, BN, BK, WM, WN, TX, TY> L;
    __shared__ __attribute__((aligned(16))) T lds_x[L::X];
    __shared__ __attribute__((aligned(16))) T lds_y[L::Y];
    __shared__ int s_task;
    for (;;) {
        if (threadIdx.x == 0) s_task = atomicAdd(counter, 1);
        __syncthreads();
        const int t = s_task;
        __syncthreads();
        if (t >= ntasks) break;
        const int2 tk = tasks[t];
        const GroupGemm<T> G = g[tk.x];
        const int64_t row0 = (int64_t)(tk.y % G.tiles_m) * BM, col0 = (int64_t)(tk.y / G.tiles_m) * BN;
        const bool interior = row0 + BM <= G.M && col0 + BN <= G.N;
        if (interior)
            gemm_tile<T, BM, BN, BK, WM, WN, TX, TY, 0, false>(G.M, G.N, G.K, G.alpha, G.X, G.ldx, G.Y, G.ldy,
                                                                   G.beta, G.C, G.ldc, row0, col0,
                                                                   (NLA_LDS T *)lds_x, (NLA_LDS T *)lds_y);
        else
            gemm_tile<T, BM, BN, BK, WM, WN, TX, TY, 0, true>(G.M, G.N, G.K, G.alpha, G.X, G.ldx, G.Y, G.ldy,
                                                                  G.beta, G.C, G.ldc, row0, col0,
                                                                  (NLA_LDS T *)lds_x, (NLA_LDS T *)lds_y);
    }
}

__global__ void zero_counter_kernel(int *p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}

// FP64: 64 x 32 tiles for side 'L', 32 x 64 for side 'R', four waves of
// 32 x 16 (16 x 32) in 16 k per step; narrow GEMMs 64 x 16 (16 x 64), four
// waves of one 16 x 16 block in 32 k per step.  FP32: 64 x 64, four waves
// of one 32 x 32 block in 32 k per step.
template <typename T, bool TX, bool TY>
static const void *gg_ptr(bool rows_m, bool narrow) {
    if constexpr (sizeof(T) == 8) {
        if (narrow) {
            if (rows_m) return (const void *)grouped_gemm_kernel<T, 64, 16, 32, 4, 1, TX, TY>;
            return (const void *)grouped_gemm_kernel<T, 16, 64, 32, 1, 4, TX, TY>;
        }
        if (rows_m) return (const void *)grouped_gemm_kernel<T, 64, 32, 16, 2, 2, TX, TY>;
        return (const void *)grouped_gemm_kernel<T, 32, 64, 16, 2, 2, TX, TY>;
    } else {
        (void)rows_m;
        (void)narrow;
        return (const void *)grouped_gemm_kernel<T, 64, 64, 32, 2, 2, TX, TY>;
    }
}

template <typename T>
const void *grouped_gemm_ptr(bool tx, bool ty, bool rows_m, bool narrow) {
    if (!tx && !ty) return gg_ptr<T, false, false>(rows_m, narrow);
    if (tx && !ty) return gg_ptr<T, true, false>(rows_m, narrow);
    if (!tx && ty) return gg_ptr<T, false, true>(rows_m, narrow);
    return gg_ptr<T, true, true>(rows_m, narrow);
}

template <typename T>
hipError_t launch_grouped_gemm(const GroupGemm<T> *g, const int2 *tasks, int ntasks, int *counter, bool tx, bool ty,
                               bool rows_m, bool narrow, int groups, hipStream_t s) {
    if (ntasks <= 0) return hipSuccess;
    hipLaunchKernelGGL(zero_counter_kernel, dim3(1), dim3(64), 0, s, counter);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    void *args[] = {(void *)&g, (void *)&tasks, (void *)&ntasks, (void *)&counter};
    return hipLaunchKernel(grouped_gemm_ptr<T>(tx, ty, rows_m, narrow), dim3(groups), dim3(256), args, 0, s);
}

template const void *grouped_gemm_ptr<float>(bool, bool, bool, bool);
template const void *grouped_gemm_ptr<double>(bool, bool, bool, bool);
template hipError_t launch_grouped_gemm<float>(const GroupGemm<float> *, const int2 *, int, int *, bool, bool, bool,
                                               bool, int, hipStream_t);
template hipError_t launch_grouped_gemm<double>(const GroupGemm<double> *, const int2 *, int, int *, bool, bool,
                                                bool, bool, int, hipStream_t);

template hipError_t launch_gemm_tiled<float>(const GemmArgs<float> &, hipStream_t);
template hipError_t launch_gemm_tiled<double>(const GemmArgs<double> &, hipStream_t);

}  // namespace nla
