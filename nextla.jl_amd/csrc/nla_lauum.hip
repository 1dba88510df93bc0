// LAUUM: A := U·U^T (uplo 'U') or L^T·L (uplo 'L') in place, only the uplo
// triangle read and written (nla_lauum in include/nla.h; the reference's
// lauum!, src/lauum.jl:52-186 with lauu2!, src/lauu2.jl:48-107).
//
// R(i,j) = sum_{k >= max(i,j)} L(k,i) L(k,j) (upper: U(i,k) U(j,k)) is one
// triangular product: a 32 x 32 (64 x 64) tile per work-group, its waves
// sharing k (nla_split_tile.h), into the caller's workspace and from there to
// A.  A tile of block row i reads the factor's rows from i down, in its own
// block and in the diagonal block of that row; so in row order, diagonal tile
// last, any run of tiles may be copied back before the next is computed, and
// the workspace of about half the triangle's size takes two to four runs.
// The recursion this replaces (a TRMM, a GEMM and a masked add per level, one
// work-group per 128-row leaf) took 2.15 ms at n = 4096 in FP64.  Up to 128
// rows are one work-group in LDS.
#include <hip/hip_runtime.h>

#include "../../include/nla.h"
#include "nla_internal.h"
#include "nla_split_tile.h"

namespace nla {

int32_t report_hip(hipError_t e, const char *where);
int32_t report_bad_arg(int k, const char *what);

namespace {

constexpr int LAUUM_LEAF = 128;  // largest diagonal block done in one work-group

// One diagonal block of nb <= NBL rows: lower R(i,j) = sum_{k>=i} L(k,i) L(k,j)
// for i >= j; upper R(i,j) = sum_{k>=j} U(i,k) U(j,k) for i <= j.  The
// triangle goes to LDS with zeros elsewhere, so every sum can run over all k
// from the block's first row; each thread owns a 4 x 4 block of R (the
// threads whose block lies outside the triangle only help load).  NBL = 64
// (256 threads) or 128 (1024 threads, 131 KB of LDS in FP64).  Both
// triangles are stored as rows of the factor the thread's index runs over
// (L(., i) for lower, U(i, .) for upper), 4 rows to a block with a stride
// of 4 NBL + 1: the 32 blocks one wave reads at a time start in 32
// different banks.
constexpr int LAUUM_RB = 4;

template <typename T, int NBL>
__global__ __launch_bounds__((NBL / 4) * (NBL / 4)) void lauum_leaf_kernel(int nb, T *__restrict__ A, int64_t lda,
                                                                        int lower) {
    constexpr int NB = NBL / LAUUM_RB, NT = NB * NB, BS = LAUUM_RB * NBL + 1;
    __shared__ T s[NB * BS];
    auto at = [](int i, int k) { return (i / LAUUM_RB) * BS + (i % LAUUM_RB) * NBL + k; };
    const int t = threadIdx.x;
    for (int e = t; e < NBL * NBL; e += NT) {
        const int r = e % NBL, c = e / NBL;
        const bool in = r < nb && c < nb && (lower ? r >= c : r <= c);
        s[lower ? at(c, r) : at(r, c)] = in ? A[r + (int64_t)c * lda] : T(0);
    }
    __syncthreads();
    const int bi = t % NB, bj = t / NB;  // rows 4 bi.., columns 4 bj..
    const int i0 = bi * LAUUM_RB, j0 = bj * LAUUM_RB;
    if ((lower ? bi < bj : bi > bj) || i0 >= nb || j0 >= nb) return;
    T acc[LAUUM_RB][LAUUM_RB];
#pragma unroll
    for (int a = 0; a < LAUUM_RB; ++a)
#pragma unroll
        for (int b = 0; b < LAUUM_RB; ++b) acc[a][b] = T(0);
    // x[a] = L(k, i0 + a) (lower) or U(i0 + a, k) (upper), zero for k below
    // the block's first row / column; y likewise for j0
    const int k0 = lower ? i0 : j0;
    for (int k = k0; k < nb; ++k) {
        T x[LAUUM_RB], y[LAUUM_RB];
#pragma unroll
        for (int a = 0; a < LAUUM_RB; ++a) {
            x[a] = s[at(i0 + a, k)];
            y[a] = s[at(j0 + a, k)];
        }
#pragma unroll
        for (int a = 0; a < LAUUM_RB; ++a)
#pragma unroll
            for (int b = 0; b < LAUUM_RB; ++b) acc[a][b] += x[a] * y[b];
    }
#pragma unroll
    for (int a = 0; a < LAUUM_RB; ++a)
#pragma unroll
        for (int b = 0; b < LAUUM_RB; ++b) {
            const int i = i0 + a, j = j0 + b;
            if (i < nb && j < nb && (lower ? i >= j : i <= j)) A[i + (int64_t)j * lda] = acc[a][b];
        }
}

// Tile p of the triangle's list: rows (lower) or columns (upper) of tiles in
// turn, the diagonal tile last in each; (i, j) with j <= i.
__device__ inline void lauum_tile(int64_t p, int64_t &i, int64_t &j) {
    i = (int64_t)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
    while (i * (i + 1) / 2 > p) --i;
    while ((i + 1) * (i + 2) / 2 <= p) ++i;
    j = p - i * (i + 1) / 2;
}

// 64 x 64 tiles (fewer operand loads per product) from LAUUM_LARGE rows on,
// 32 x 32 below, where they are too few for the chip.  Measured on MI355X (us,
// 32 / 64, lower): FP64 n = 2048 133 / 150, 3000 250 / 262, 4096 715 / 511,
// 8192 5026 / 3144 (58 TFLOP/s); FP32 3000 159 / 149, 4096 367 / 263, 8192
// 2532 / 1671.
constexpr int LAUUM_KS = 4;
constexpr int64_t LAUUM_LARGE = 3072;

// Tiles p0 + blockIdx of R into W, B x B each (B = 16 RB).
template <typename T, int RB, bool LOWER>
__global__ __launch_bounds__(LAUUM_KS * 64) void lauum_product_kernel(int64_t n, const T *__restrict__ A, int64_t lda,
                                                                      T *__restrict__ W, int64_t p0) {
    constexpr int B = 16 * RB;
    __shared__ T red[LAUUM_KS * RB * RB * 4 * 64];
    int64_t i, j;
    lauum_tile(p0 + blockIdx.x, i, j);
    const int64_t row0 = (LOWER ? i : j) * B, col0 = (LOWER ? j : i) * B;
    T *C = W + (int64_t)blockIdx.x * B * B;
    // lower: op(X)(i,k) = L(k,i), op(Y)(k,j) = L(k,j); upper: U(i,k), U(j,k)
    if (row0 + B <= n && col0 + B <= n)
        split_tile<T, RB, RB, LAUUM_KS, LOWER, !LOWER, false, true>(n, n, n, T(1), A, lda, A, lda, T(0), C, B, row0,
                                                                    col0, (NLA_LDS T *)red);
    else
        split_tile<T, RB, RB, LAUUM_KS, LOWER, !LOWER, true, true>(n, n, n, T(1), A, lda, A, lda, T(0), C, B, row0,
                                                                   col0, (NLA_LDS T *)red);
}

// The same tiles from W to A's triangle.
template <typename T, int B, bool LOWER>
__global__ __launch_bounds__(256) void lauum_store_kernel(int64_t n, T *__restrict__ A, int64_t lda,
                                                          const T *__restrict__ W, int64_t p0) {
    int64_t i, j;
    lauum_tile(p0 + blockIdx.x, i, j);
    const int64_t row0 = (LOWER ? i : j) * B, col0 = (LOWER ? j : i) * B;
    const T *w = W + (int64_t)blockIdx.x * B * B;
    const int64_t r = row0 + threadIdx.x % B;
    for (int64_t c = col0 + threadIdx.x / B; c < col0 + B; c += 256 / B)
        if (r < n && c < n && (LOWER ? r >= c : r <= c)) A[r + c * lda] = w[(r - row0) + (c - col0) * B];
}

template <typename T, int RB, bool LOWER>
hipError_t lauum_product(int64_t n, T *A, int64_t lda, T *W, int64_t elems, hipStream_t s) {
    constexpr int64_t B = 16 * RB;
    const int64_t t = (n + B - 1) / B, total = t * (t + 1) / 2, cap = elems / (B * B);
    for (int64_t p = 0; p < total; p += cap) {
        const unsigned g = (unsigned)(total - p < cap ? total - p : cap);
        hipLaunchKernelGGL((lauum_product_kernel<T, RB, LOWER>), dim3(g), dim3(LAUUM_KS * 64), 0, s, n, A, lda, W, p);
        hipLaunchKernelGGL((lauum_store_kernel<T, (int)B, LOWER>), dim3(g), dim3(256), 0, s, n, A, lda, W, p);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename T>
int32_t lauum_typed(bool lower, int64_t n, T *A, int64_t lda, T *W, int64_t elems, hipStream_t s) {
    hipError_t e;
    if (n <= LAUUM_LEAF) {
        if (n <= 64)
            hipLaunchKernelGGL((lauum_leaf_kernel<T, 64>), dim3(1), dim3(256), 0, s, (int)n, A, lda, lower ? 1 : 0);
        else
            hipLaunchKernelGGL((lauum_leaf_kernel<T, 128>), dim3(1), dim3(1024), 0, s, (int)n, A, lda, lower ? 1 : 0);
        e = hipGetLastError();
    } else if (n >= LAUUM_LARGE) {
        e = lower ? lauum_product<T, 4, true>(n, A, lda, W, elems, s) : lauum_product<T, 4, false>(n, A, lda, W, elems, s);
    } else {
        e = lower ? lauum_product<T, 2, true>(n, A, lda, W, elems, s) : lauum_product<T, 2, false>(n, A, lda, W, elems, s);
    }
    return e == hipSuccess ? NLA_OK : report_hip(e, "lauum");
}

}  // namespace
}  // namespace nla

using namespace nla;

extern "C" {

int64_t nla_lauum_workspace_bytes(int32_t dtype, int64_t n) {
    if ((dtype != NLA_F32 && dtype != NLA_F64) || n < 0) return -1;
    const int64_t h = ((n / 2 + 63) / 64) * 64;
    return (n > LAUUM_LEAF ? h * h : 1) * (dtype == NLA_F64 ? 8 : 4);
}

int32_t nla_lauum(char uplo, int32_t dtype, int64_t n, void *A, int64_t lda, void *workspace,
                  int64_t workspace_bytes, void *stream) {
    uplo = (uplo == 'l') ? 'L' : (uplo == 'u') ? 'U' : uplo;
    if (uplo != 'L' && uplo != 'U') return report_bad_arg(1, "uplo");
    if (dtype != NLA_F32 && dtype != NLA_F64) return report_bad_arg(2, "dtype");
    if (n < 0) return report_bad_arg(3, "n");
    if (n > 0 && A == nullptr) return report_bad_arg(4, "A");
    if (lda < (n > 1 ? n : 1)) return report_bad_arg(5, "lda");
    const int64_t need = nla_lauum_workspace_bytes(dtype, n);
    if (n > LAUUM_LEAF && (workspace == nullptr || workspace_bytes < need)) return report_bad_arg(7, "workspace_bytes");
    if (n == 0) return NLA_OK;
    hipStream_t s = (hipStream_t)stream;
    const int64_t h = ((n / 2 + 63) / 64) * 64;
    return dtype == NLA_F64 ? lauum_typed<double>(uplo == 'L', n, (double *)A, lda, (double *)workspace, h * h, s)
                            : lauum_typed<float>(uplo == 'L', n, (float *)A, lda, (float *)workspace, h * h, s);
}

}  // extern "C"
