// One tile of a product by a work-group whose KS waves share K, loading their
// operands straight into registers: the GEMM update where tiles are few
// (nla_gemm_split.hip) and lauum's product (nla_lauum.hip).
//
// Every wave multiplies the whole tile over its own range of k, three 16-deep
// blocks ahead, and the waves' partial tiles meet in LDS, added in a fixed
// order.  No wave waits for another before that.
//
// Operand layout.  MFMA steps may take any k, as long as both operands take
// the same one: step s of a 16-deep block uses k = 4 (lane / 16) + s, so a
// k-contiguous operand is loaded four elements at a time.  An operand that
// is contiguous along its outer index is loaded two elements at a time, its
// 16-blocks in pairs with block b holding the outer indices of parity b.
// Loads need no more than an element's alignment (global memory takes
// unaligned 16-byte loads), so odd leading dimensions cost nothing here.
#pragma once

#include <limits>

#include "nla_device.h"

namespace nla {

typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
typedef float f2u_t __attribute__((ext_vector_type(2), aligned(4)));
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

#ifndef NLA_LDS
#define NLA_LDS __attribute__((address_space(3)))
#endif

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
    // zero what lies before the diagonal: keep k >= outer; d: the outer origin
    // minus the block's first k
    __device__ static inline void keep_upper(T (*v)[4], int d, int lane) {
        const int lo = lane & 15, kk = 4 * (lane >> 4);
#pragma unroll
        for (int b = 0; b < NBK; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) v[b][s] = kk + s >= d + outer(b, lo) ? v[b][s] : T(0);
    }
};

// C's tile at (row0, col0) = beta*C + alpha*op(X)*op(Y); C: the tile's first
// element.  EDGE: the tile may reach past M or N.  TRI: op(X)(i, k) and
// op(Y)(k, j) count only where k >= i and k >= j, whatever is stored elsewhere.
template <typename T, int RB, int CB, int KS, bool TX, bool TY, bool EDGE, bool TRI = false>
__device__ __forceinline__ void split_tile(int64_t M, int64_t N, int64_t K, T alpha, const T *__restrict__ X,
                                           int64_t ldx, const T *__restrict__ Y, int64_t ldy, T beta,
                                           T *__restrict__ C, int64_t ldc, int64_t row0, int64_t col0,
                                           NLA_LDS T *red) {
    typedef SplitMma<T> MM;
    typedef SplitOperand<T, RB, TX, EDGE> OX;
    typedef SplitOperand<T, CB, !TY, EDGE> OY;
    constexpr int NR = RB * CB * 4, PD = 3;  // registers of a partial tile; blocks in flight
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t k0 = TRI ? (row0 > col0 ? row0 : col0) : 0, nfull = (K - k0) / 16;
    const int tail = (int)((K - k0) % 16);
    const int64_t b0 = nfull * w / KS, b1 = nfull * (w + 1) / KS;
    typename MM::acc_t acc[CB][RB];
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < RB; ++r) acc[c][r] = typename MM::acc_t{T(0), T(0), T(0), T(0)};
    OX ox;
    OY oy;
    ox.init(X, ldx, row0, M, k0 + 16 * b0, lane);
    oy.init(Y, ldy, col0, N, k0 + 16 * b0, lane);
    T xv[PD][RB][4], yv[PD][CB][4];
    // block b of this wave, in registers u
    auto mul = [&](int64_t b, int u) {
        if constexpr (TRI) {  // only the blocks beside the diagonal hold anything to drop
            const int64_t k = k0 + 16 * (b0 + b);
            if (k < row0 + 16 * RB) OX::keep_upper(xv[u], (int)(row0 - k), lane);
            if (k < col0 + 16 * CB) OY::keep_upper(yv[u], (int)(col0 - k), lane);
        }
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
                mul(b + u, u);
            }
        }
#pragma unroll
        for (int u = 0; u < PD - 1; ++u)
            if (b + u < nb) mul(b + u, u);
    }
    if (tail != 0 && w == KS - 1) {
        ox.init(X, ldx, row0, M, k0 + 16 * nfull, lane);
        oy.init(Y, ldy, col0, N, k0 + 16 * nfull, lane);
        ox.load_tail(xv[0], tail, lane);
        oy.load_tail(yv[0], tail, lane);
        mul(nfull - b0, 0);
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
        const int tr = OX::outer(r, lane & 15), tc = OY::outer(c, MM::di(lane, e));
        in[i] = !EDGE || (row0 + tr < M && col0 + tc < N);
        d[i] = in[i] ? C + tr + tc * ldc : C;
        cv[i] = beta == T(0) ? T(0) : beta * *d[i];
    }
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[(w * NR + (c * RB + r) * 4 + e) * 64 + lane] = acc[c][r][e];
    __syncthreads();
    bool odd = false;
#pragma unroll
    for (int i = 0; i < NR / KS; ++i) {
        const int q = i * KS + w;
        T sum = red[q * 64 + lane];
#pragma unroll
        for (int v = 1; v < KS; ++v) sum += red[(v * NR + q) * 64 + lane];
        if (TRI) odd |= !(fabs(sum) <= std::numeric_limits<T>::max());
        if (in[i]) *d[i] = alpha * sum + cv[i];
    }
    if constexpr (TRI) {
        // a zero that stands for one operand's other triangle, times an
        // infinity or NaN of the other: such sums again, over their own k
        // (beta is 0 here)
        if (odd) {
#pragma unroll 1
            for (int q = w; q < NR; q += KS) {
                const int64_t r = OX::outer(q / 4 % RB, lane & 15), c = OY::outer(q / (4 * RB), MM::di(lane, q % 4));
                if (row0 + r >= M || col0 + c >= N) continue;
                T *p = C + r + c * ldc;
                if (fabs(*p) <= std::numeric_limits<T>::max()) continue;
                const T *x = X + (TX ? (row0 + r) * ldx : row0 + r), *y = Y + (TY ? col0 + c : (col0 + c) * ldy);
                T sum = T(0);
#pragma unroll 1
                for (int64_t k = row0 + r > col0 + c ? row0 + r : col0 + c; k < K; ++k)
                    sum += x[TX ? k : k * ldx] * y[TY ? k * ldy : k];
                *p = alpha * sum;
            }
        }
    }
}

}  // namespace nla
