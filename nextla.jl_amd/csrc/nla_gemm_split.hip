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
// every wave multiplies the whole tile over its own range of k with operands
// loaded straight into registers, three 16-deep blocks ahead, and the waves'
// partial tiles meet in LDS, added in a fixed order.  No wave waits for
// another before that.
//
// Operand layout.  MFMA steps may take any k, as long as both operands take
// the same one: step s of a 16-deep block uses k = 4 (lane / 16) + s, so a
// k-contiguous operand is loaded four elements at a time.  An operand that
// is contiguous along its outer index is loaded two elements at a time, its
// 16-blocks in pairs with block b holding the outer indices of parity b.
// Loads need no more than an element's alignment (global memory takes
// unaligned 16-byte loads), so odd leading dimensions cost nothing here.
#include "nla_device.h"
#include "nla_internal.h"

namespace nla {

namespace {

typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
typedef float f2u_t __attribute__((ext_vector_type(2), aligned(4)));
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

#define NLA_LDS __attribute__((address_space(3)))

template <typename T>
struct SplitMma;
template <>
struct SplitMma<double> {
    typedef d4_t acc_t;
    typedef d2u_t v2_t;
    __device__ static inline acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static inline int di(int l, int r) { return 4 * r + (l >> 4); }
    __device__ static inline void load4(const double *p, double *v) {
        const d2u_t a = *(const d2u_t *)p, b = *(const d2u_t *)(p + 2);
        v[0] = a[0];
        v[1] = a[1];
        v[2] = b[0];
        v[3] = b[1];
    }
};
template <>
struct SplitMma<float> {
    typedef f4_t acc_t;
    typedef f2u_t v2_t;
    __device__ static inline acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static inline int di(int l, int r) { return 4 * (l >> 4) + r; }
    __device__ static inline void load4(const float *p, float *v) {
        const f4u_t a = *(const f4u_t *)p;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = a[i];
    }
};

// One operand of a wave's tile: NBK blocks of 16 outer indices from o0, k
// blocks of 16.  KC: contiguous along k.  EDGE: outer indices past no - 1
// read no - 1 (their results are not stored).
template <typename T, int NBK, bool KC, bool EDGE>
struct SplitOperand {
    typedef SplitMma<T> MM;
    static constexpr bool PAIR = !KC && NBK % 2 == 0;
    // pointers to this lane's first element of each block (k = 4 (lane / 16))
    const T *p[NBK];
    int64_t ld;

    // outer index of (block b, lane l % 16)
    __device__ static inline int outer(int b, int lo) {
        return PAIR ? (b >> 1) * 32 + 2 * lo + (b & 1) : b * 16 + lo;
    }
    __device__ inline void init(const T *P, int64_t ld_, int64_t o0, int64_t no, int64_t k0, int lane) {
        ld = ld_;
        const int lo = lane & 15, kk = 4 * (lane >> 4);
#pragma unroll
        for (int b = 0; b < NBK; ++b) {
            int64_t o = o0 + outer(b, lo);
            if (EDGE) o = o < no ? o : no - 1;
            p[b] = KC ? P + o * ld + (k0 + kk) : P + o + (k0 + kk) * ld;
        }
    }
    // the 16-deep block at the pointers, which then move on by step blocks
    __device__ inline void load(T (*v)[4], int64_t step) {
        if constexpr (KC) {
#pragma unroll
            for (int b = 0; b < NBK; ++b) {
                MM::load4(p[b], v[b]);
                p[b] += 16 * step;
            }
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if constexpr (PAIR && !EDGE) {
#pragma unroll
                    for (int b = 0; b < NBK; b += 2) {
                        const typename MM::v2_t a = *(const typename MM::v2_t *)(p[b] + s * ld);
                        v[b][s] = a[0];
                        v[b + 1][s] = a[1];
                    }
                } else {
#pragma unroll
                    for (int b = 0; b < NBK; ++b) v[b][s] = p[b][s * ld];
                }
            }
#pragma unroll
            for (int b = 0; b < NBK; ++b) p[b] += 16 * step * ld;
        }
    }
    // the last, partial block: nk (1..15) valid k from the block's start
    __device__ inline void load_tail(T (*v)[4], int nk, int lane) {
        const int kk = 4 * (lane >> 4);
#pragma unroll
        for (int b = 0; b < NBK; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const bool ok = kk + s < nk;
                // past the end: the block's first k of this outer index (valid)
                const int64_t d = ok ? s : -kk;
                const T x = p[b][KC ? d : d * ld];
                v[b][s] = ok ? x : T(0);
            }
    }
};

template <typename T, int RB, int CB, int KS, bool TX, bool TY, bool EDGE>
__device__ __forceinline__ void split_tile(int64_t M, int64_t N, int64_t K, T alpha, const T *__restrict__ X,
                                           int64_t ldx, const T *__restrict__ Y, int64_t ldy, T beta,
                                           T *__restrict__ C, int64_t ldc, int64_t row0, int64_t col0,
                                           NLA_LDS T *red) {
    typedef SplitMma<T> MM;
    typedef SplitOperand<T, RB, TX, EDGE> OX;
    typedef SplitOperand<T, CB, !TY, EDGE> OY;
    constexpr int NR = RB * CB * 4, PD = 3;  // registers of a partial tile; blocks in flight
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t nfull = K / 16;
    const int tail = (int)(K % 16);
    const int64_t b0 = nfull * w / KS, b1 = nfull * (w + 1) / KS;
    typename MM::acc_t acc[CB][RB];
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < RB; ++r) acc[c][r] = typename MM::acc_t{T(0), T(0), T(0), T(0)};
    OX ox;
    OY oy;
    ox.init(X, ldx, row0, M, 16 * b0, lane);
    oy.init(Y, ldy, col0, N, 16 * b0, lane);
    T xv[PD][RB][4], yv[PD][CB][4];
    auto mul = [&](int u) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int r = 0; r < RB; ++r) acc[c][r] = MM::mma(yv[u][c][s], xv[u][r][s], acc[c][r]);
    };
    // a ring of PD register blocks; loads past the wave's range are its last
    // block again (no load under a branch: the compiler would wait for it at
    // the join)
    const int nb = (int)(b1 - b0);
    if (nb > 0) {
#pragma unroll
        for (int u = 0; u < PD - 1; ++u) {
            const int64_t step = u + 1 < nb ? 1 : 0;
            ox.load(xv[u], step);
            oy.load(yv[u], step);
        }
        int b = 0;
        for (; b + PD <= nb; b += PD) {
#pragma unroll
            for (int u = 0; u < PD; ++u) {
                const int64_t step = b + u + PD < nb ? 1 : 0;
                ox.load(xv[(u + PD - 1) % PD], step);
                oy.load(yv[(u + PD - 1) % PD], step);
                mul(u);
            }
        }
#pragma unroll
        for (int u = 0; u < PD - 1; ++u)
            if (b + u < nb) mul(u);
    }
    if (tail != 0 && w == KS - 1) {
        ox.init(X, ldx, row0, M, 16 * nfull, lane);
        oy.init(Y, ldy, col0, N, 16 * nfull, lane);
        ox.load_tail(xv[0], tail, lane);
        oy.load_tail(yv[0], tail, lane);
        mul(0);
    }
    // partial tiles: register q of wave w at red[(w * NR + q) * 64 + lane];
    // wave w then adds registers w, w + KS, ... of all waves, in wave order.
    // C's own values are requested before the waves meet.
    static_assert(NR % KS == 0, "registers divide among the waves");
    T *d[NR / KS];
    T cv[NR / KS];
    bool in[NR / KS];
#pragma unroll
    for (int i = 0; i < NR / KS; ++i) {
        const int q = i * KS + w, c = q / (4 * RB), r = q / 4 % RB, e = q % 4;
        const int64_t row = row0 + OX::outer(r, lane & 15), col = col0 + OY::outer(c, MM::di(lane, e));
        in[i] = !EDGE || (row < M && col < N);
        d[i] = in[i] ? C + row + col * ldc : C;
        cv[i] = beta == T(0) ? T(0) : beta * *d[i];
    }
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[(w * NR + (c * RB + r) * 4 + e) * 64 + lane] = acc[c][r][e];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NR / KS; ++i) {
        const int q = i * KS + w;
        T sum = red[q * 64 + lane];
#pragma unroll
        for (int v = 1; v < KS; ++v) sum += red[(v * NR + q) * 64 + lane];
        if (in[i]) *d[i] = alpha * sum + cv[i];
    }
}

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
        split_tile<T, RB, CB, KS, TX, TY, false>(M, N, K, alpha, X, ldx, Y, ldy, beta, C, ldc, row0, col0,
                                                 (NLA_LDS T *)red);
    else
        split_tile<T, RB, CB, KS, TX, TY, true>(M, N, K, alpha, X, ldx, Y, ldy, beta, C, ldc, row0, col0,
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
    // tiles were within 10 % of 32 x 32 with four or slower.
    if (a.leaf == 0 && a.tri == 0 && a.K > 0) {
        auto tiles = [&](int b) { return ((a.M + b - 1) / b) * ((a.N + b - 1) / b); };
        const bool split = sizeof(T) == 8 ? tiles(128) <= (a.K < 128 ? 64 : 192) : tiles(64) <= 144;
        if (split) return launch_split<T, 2, 2, 4>(a, s);
    }
    return launch_gemm_tiled<T>(a, s);
}

template hipError_t launch_gemm<float>(const GemmArgs<float> &, hipStream_t);
template hipError_t launch_gemm<double>(const GemmArgs<double> &, hipStream_t);

}  // namespace nla
