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
    // Split where few tiles leave the chip idle (`idle`; past it, as at 30000 x
    // 32 x 1000 in FP64 where a split would take 49 us for 134, products keep the
    // order of the tiles' sums) and its estimated time is the shorter: q tiles of
    // 32 x 32 per CU, each with a start and end of 0.6 us and the rate of its
    // orientation (with op(X) transposed a lane loads from 16 rows of memory),
    // against the rounds of the tiled kernels and the 1.6 us that their first and
    // last steps take more. Measured on MI355X (us per launch, tiled / split):
    // FP64 64 x 4096 x 4096 371 / 50, 1024^3 90 / 49, 1280 x 1280 x 512 49 / 42,
    // 1408 x 1408 x 192 22.9 / 30.2, 1024 x 1024 x 48 9.3 / 10.0, with X
    // transposed 9.3 / 12.2, 1152 x 1152 x 192 so 21.4 / 30.5, 1024 x 1024 x 1024
    // so 88 / 64; FP32 512 x 512 x 192 6.6 / 4.8, 768 x 768 x 64 4.8 / 5.5, 704 x
    // 704 x 1024 24 / 16. At most 10 % from the faster one over K = 16 .. 4096
    // and 16 to 4096 tiles of 32 x 32, 0.5 % on average.
    if (a.leaf == 0 && a.tri == 0 && a.K > 0) {
        constexpr bool F64 = sizeof(T) == 8;
        auto tiles = [&](int b) { return ((a.M + b - 1) / b) * ((a.N + b - 1) / b); };
        const bool idle = F64 ? tiles(128) <= (a.K < 128 ? 64 : (a.tx ? 96 : 192)) : tiles(64) <= 144;
        const int64_t q = (tiles(32) + 255) / 256;
        const double rate = F64 ? (a.tx ? (a.ty ? 0.0104 : 0.0150) : (a.ty ? 0.0090 : 0.0094))
                                : (a.tx ? (a.ty ? 0.0070 : 0.0074) : 0.0062);  // us per k and tile of a CU
        double tiled = 0;
        gemm_tile_shape<T>(a.M, a.N, (a.K + 15) / 16 * 16, &tiled);
        if (idle && (double)q * (0.6 + rate * (double)(a.K + (F64 ? 16 : 32))) < tiled + 1.6)
            return launch_split<T, 2, 2, 4>(a, s);
    }
    return launch_gemm_tiled<T>(a, s);
}

template hipError_t launch_gemm<float>(const GemmArgs<float> &, hipStream_t);
template hipError_t launch_gemm<double>(const GemmArgs<double> &, hipStream_t);

}  // namespace nla
