// GEMM update for shapes whose tiles do not fill the chip, and the choice
// between it and the tiled kernels of nla_gemm.hip.
//
//   C = beta*C + alpha*op(X)*op(Y)      op(X): M x K, op(Y): K x N, C: M x N
//
// Replaces matmul! (src/matmul.jl:5-66) where a block of the recursion, a
// panel update with few right-hand sides or a block reflector's inner product
// gives fewer 64 x 128 tiles than the card has compute units.
//
// What bounds such a product is latency: few work-groups, each walking all of
// K.  Here a work-group owns a 32 x 32 tile and its KS = 4 waves share K:
// no wave waits for another before the end (nla_split_tile.h).
#include "nla_internal.h"
#include "nla_split_tile.h"

namespace nla {

namespace {

template <typename T, int RB, int CB, int KS, bool TX, bool TY>
__global__ __launch_bounds__(KS * 64) void gemm_split_kernel(int64_t M, int64_t N, int64_t K, T alpha,
                                                             const T *__restrict__ X, int64_t ldx,
                                                             const T *__restrict__ Y, int64_t ldy, T beta,
                                                             T *__restrict__ C, int64_t ldc, int tiles_m) {
    __shared__ T red[KS * RB * CB * 4 * 64];
    // work-group g runs on XCD g % 8: each XCD takes a contiguous range of
    // tiles, down the columns, so that they share Y's columns in its L2
    const int G = (int)gridDim.x, g = (int)blockIdx.x;
    const int xcd = g % 8, idx = g / 8, per = G / 8, rem = G % 8;
    const int gp = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
    const int64_t row0 = (int64_t)(gp % tiles_m) * (16 * RB), col0 = (int64_t)(gp / tiles_m) * (16 * CB);
    if (row0 + 16 * RB <= M && col0 + 16 * CB <= N)
        split_tile<T, RB, CB, KS, TX, TY, false>(M, N, K, alpha, X, ldx, Y, ldy, beta, C + row0 + col0 * ldc, ldc, row0, col0,
                                                 (NLA_LDS T *)red);
    else
        split_tile<T, RB, CB, KS, TX, TY, true>(M, N, K, alpha, X, ldx, Y, ldy, beta, C + row0 + col0 * ldc, ldc, row0, col0,
                                                (NLA_LDS T *)red);
}

template <typename T, int RB, int CB, int KS>
hipError_t launch_split(const GemmArgs<T> &a, hipStream_t s) {
    const int64_t tm = (a.M + 16 * RB - 1) / (16 * RB), tn = (a.N + 16 * CB - 1) / (16 * CB);
    const dim3 grid((unsigned)(tm * tn)), block(KS * 64);
#define NLA_SPLIT(TX, TY)                                                                                            \
    hipLaunchKernelGGL((gemm_split_kernel<T, RB, CB, KS, TX, TY>), grid, block, 0, s, a.M, a.N, a.K, a.alpha, a.X,   \
                       a.ldx, a.Y, a.ldy, a.beta, a.C, a.ldc, (int)tm)
    if (!a.tx && !a.ty) NLA_SPLIT(false, false);
    else if (a.tx && !a.ty) NLA_SPLIT(true, false);
    else if (!a.tx) NLA_SPLIT(false, true);
    else NLA_SPLIT(true, true);
#undef NLA_SPLIT
    return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t launch_gemm(const GemmArgs<T> &a, hipStream_t s) {
    if (a.M <= 0 || a.N <= 0) return hipSuccess;
    // Measured on MI355X (us per launch, tiled / split): FP64 512^3 (K = 256)
    // 28.7 / 7.1, 1024 x 1024 x 1024 103 / 47, 64 x 4096 x 4096 390 / 40,
    // 4096 x 8 x 4096 523 / 38, 3000 x 1000 x 512 105 / 69, 1792 x 1792 x 256
    // 47 / 48, 2048 x 2048 x 256 45 / 60, and with K = 64, where C's traffic
    // counts, 1024 x 1024 11.8 / 11.6, 1280 x 1280 12.4 / 15.2.  FP32, whose
    // smallest tile is 64 x 64: 512 x 512 x 256 9.2 / 5.4, 768 x 768 x 1024
    // 26.8 / 21.7, 1024 x 1024 x 256 10.2 / 11.8, 64 x 4096 x 4096 97 / 31,
    // 256 x 4096 x 4096 101 / 100.  Eight waves per tile, 64 x 16 and 64 x 64
    // tiles were within 10 % of 32 x 32 with four or slower.  FP64 with op(X)
    // transposed, whose lanes load from 16 rows of memory, reaches 36 TFLOP/s
    // here (48 otherwise): a block reflector of 8192 x 8192 with k = 256, 128
    // tiles, takes 1453 / 1700 us tiled / split.
    if (a.leaf == 0 && a.tri == 0 && a.K > 0) {
        auto tiles = [&](int b) { return ((a.M + b - 1) / b) * ((a.N + b - 1) / b); };
        const bool split = sizeof(T) == 8 ? tiles(128) <= (a.K < 128 ? 64 : (a.tx ? 96 : 192)) : tiles(64) <= 144;
        if (split) return launch_split<T, 2, 2, 4>(a, s);
    }
    return launch_gemm_tiled<T>(a, s);
}

template hipError_t launch_gemm<float>(const GemmArgs<float> &, hipStream_t);
template hipError_t launch_gemm<double>(const GemmArgs<double> &, hipStream_t);

}  // namespace nla
