// Diagonal-block leaves of the recursive triangular solve / multiply.
//
// Replaces the eight reference leaf kernels: lower_left_kernel,
// upper_left_kernel, right_lower_kernel, right_upper_kernel (src/trsm.jl:5-126)
// and Left/Right{Lower,Upper}TRMM_kernel! (src/trmm.jl:43-312).
//
// All eight (side, uplo) forms, with or without transpose, are reduced to one
// canonical problem on a lower-triangular nb x nb block L:
//   TRSM:  L * X = pre * Bc        (forward substitution)
//   TRMM:  Bc <- post * (L * Bc)
// with L(i, j) = A[i*ars + j*acs] and Bc(i, c) = B[i*brs + c*bcs].  Upper
// triangles are made lower by the reversal permutation (negative strides from
// the last diagonal element), and right-side problems are solved on the
// transpose (X*op(A) = B  <=>  op(A)^T X^T = B^T), so the caller only picks
// pointers and signed strides.
//
// Each lane owns one right-hand-side column and keeps all NB of its entries in
// registers; the block of L sits in LDS and is read with wave-uniform
// addresses (one broadcast LDS read serves all 64 lanes), so the sweep has no
// barriers at all (the reference takes one barrier per row, src/trsm.jl:21-27).
// The RHS tile is staged through LDS so that HBM is always walked along its
// contiguous direction (down columns for the left side, along rows for the
// right side) whatever the lane-to-column mapping.
#include "nla_device.h"
#include "nla_internal.h"

namespace nla {

constexpr int LEAF_COLS = 64;  // RHS columns per work-group (one per lane)

// ICONTIG: Bc is contiguous along i (left side) rather than along c (right
// side); the RHS tile is staged through LDS either way, walking the
// contiguous direction so every wave-wide load and store is coalesced.
template <typename T, int NB, bool ICONTIG, bool TRMM>
__global__ __launch_bounds__(LEAF_COLS) void leaf_kernel(int nb, int64_t m, const T *__restrict__ A, int64_t ars,
                                                         int64_t acs, T *__restrict__ B, int64_t brs, int64_t bcs,
                                                         T scale) {
    // TRSM reads L by columns (column j after x[j] is final), TRMM by rows
    // (row i is a dot product over j <= i); store L in the matching order.
    __shared__ __attribute__((aligned(16))) T sl[NB * NB];
    __shared__ T srinv[NB];
    __shared__ T sb[LEAF_COLS * (NB + 1)];

    const int t = threadIdx.x;
    const int64_t c0 = (int64_t)blockIdx.x * LEAF_COLS;

    // Stage L, padded to NB with an identity block.  Loads are issued in
    // batches of SB before any LDS write so HBM/L2 latency overlaps.
    constexpr int SB = 16;
    const bool arow = (ars == 1 || ars == -1);  // walk the contiguous direction
#pragma unroll 1
    for (int e0 = 0; e0 < NB * NB; e0 += SB * LEAF_COLS) {
        T v[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            int e = e0 + u * LEAF_COLS + t;
            int i = arow ? e % NB : e / NB;
            int j = arow ? e / NB : e % NB;
            bool in = e < NB * NB;
            if (in && i < nb && j < nb)
                v[u] = (j <= i) ? A[i * ars + j * acs] : T(0);
            else
                v[u] = (i == j) ? T(1) : T(0);
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            int e = e0 + u * LEAF_COLS + t;
            int i = arow ? e % NB : e / NB;
            int j = arow ? e / NB : e % NB;
            if (e < NB * NB) {
                if (TRMM)
                    sl[i * NB + j] = v[u];
                else
                    sl[j * NB + i] = v[u];
            }
        }
    }
    if (!TRMM) {
        for (int i = t; i < NB; i += LEAF_COLS) srinv[i] = (i < nb) ? T(1) / A[i * ars + i * acs] : T(1);
    }

    // Load this lane's column of Bc.
    T x[NB];
#pragma unroll 1
    for (int e0 = 0; e0 < NB * LEAF_COLS; e0 += SB * LEAF_COLS) {
        T v[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            int e = e0 + u * LEAF_COLS + t;
            int i = ICONTIG ? e % NB : e / LEAF_COLS;
            int c = ICONTIG ? e / NB : e % LEAF_COLS;
            int64_t gc = c0 + c;
            v[u] = (i < nb && gc < m) ? B[i * brs + gc * bcs] : T(0);
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            int e = e0 + u * LEAF_COLS + t;
            int i = ICONTIG ? e % NB : e / LEAF_COLS;
            int c = ICONTIG ? e / NB : e % LEAF_COLS;
            sb[c * (NB + 1) + i] = v[u];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) x[i] = sb[t * (NB + 1) + i];

    if (!TRMM) {
        // alpha of unified_rectrxm! (src/rectrxm.jl:64) applied on first touch.
        if (scale != T(1)) {
#pragma unroll
            for (int i = 0; i < NB; ++i) x[i] *= scale;
        }
        // Forward substitution, column oriented: once x[j] is final, remove
        // its contribution from every later row.
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            x[j] = x[j] * srinv[j];
#pragma unroll
            for (int r = j + 1; r < NB; ++r) x[r] = x[r] - sl[j * NB + r] * x[j];
        }
    } else {
        // Triangular product in place: row i needs the original x[0..i], so
        // rows are formed from the bottom up.
#pragma unroll
        for (int i = NB - 1; i >= 0; --i) {
            T s = T(0);
#pragma unroll
            for (int j = 0; j <= i; ++j) s += sl[i * NB + j] * x[j];
            x[i] = scale * s;
        }
    }

#pragma unroll
    for (int i = 0; i < NB; ++i) sb[t * (NB + 1) + i] = x[i];
    __syncthreads();
#pragma unroll 16
    for (int e = t; e < NB * LEAF_COLS; e += LEAF_COLS) {
        int i = ICONTIG ? e % NB : e / LEAF_COLS;
        int c = ICONTIG ? e / NB : e % LEAF_COLS;
        int64_t gc = c0 + c;
        if (i < nb && gc < m) B[i * brs + gc * bcs] = sb[c * (NB + 1) + i];
    }
}

// 16 x 16 x 4 MFMA: step s of a lane in group kk = lane / 16 takes k =
// kmap(kk, s), which is also the row of its result register s.
template <typename T>
struct Mma16;
template <>
struct Mma16<double> {
    typedef d4_t acc_t;
    __device__ static inline acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static inline int kmap(int kk, int s) { return 4 * s + kk; }
    static constexpr double big = 0x1p500;
};
template <>
struct Mma16<float> {
    typedef f4_t acc_t;
    __device__ static inline acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static inline int kmap(int kk, int s) { return 4 * kk + s; }
    static constexpr float big = 0x1p60f;
};

// Inverse of one 64 x 64 triangular block with 256 threads, in three stages
// (the blocked scheme of LAPACK's trtri), in place in LDS:
//   1. the four 16 x 16 diagonal sub-blocks by substitution on the columns of
//      the identity (64 lanes, one column each, 16-step chains);
//   2. 32 x 32 inverses: inv([A 0; C B]) = [inv A, 0; -inv B * C * inv A, inv B],
//      on MFMA, the result written over C;
//   3. the same step from 32 to 64.
// sl: the canonical lower block (column-major, leading dimension TRTRI_LD),
// which becomes its inverse; sp: TRTRI_SP scratch.  The parts above the
// diagonal stay zero, so the products run over full k ranges and the extra
// terms add exact zeros.  Upper blocks are inverted as J U J.  A call of one
// block is bound by its chain (loads, 16 quotients, two product stages), the
// batched form by LDS traffic: with the products in FMAs a thread read two
// LDS words per multiply.  38 KB of LDS in FP64, four work-groups per CU.
constexpr int TRTRI_LD = 66, TRTRI_SP = 576;
template <typename T>
__device__ __forceinline__ void trtri64_block(int64_t n, int64_t blk, const T *__restrict__ A, int64_t rs, int64_t cs, bool lower,
                              bool unit, T *__restrict__ W, T *sl, T *sp, int *__restrict__ F) {
    constexpr int NB = 64, NT = 256, LD = TRTRI_LD;
    const int t = threadIdx.x;
    const int64_t off = blk * NB;
    const int nb = (int)(n - off < NB ? n - off : NB);
    const T *base = lower ? A + off * (rs + cs) : A + (off + nb - 1) * (rs + cs);
    const int64_t ars = lower ? rs : -rs, acs = lower ? cs : -cs;
    const bool arow = (ars == 1 || ars == -1);
    // stage L (identity padding past nb).  All 16 loads of a thread are
    // issued before the first LDS store.
    constexpr int PER = NB * NB / NT;
    T v[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int e = t + u * NT;
        const int i = arow ? e % NB : e / NB;
        const int j = arow ? e / NB : e % NB;
        // a unit diagonal is taken as 1 and not read
        const bool ok = i < nb && j < nb && j <= i && !(unit && i == j);
        v[u] = *(ok ? base + i * ars + j * acs : base);
        v[u] = ok ? v[u] : (i == j ? T(1) : T(0));
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int e = t + u * NT;
        const int i = arow ? e % NB : e / NB;
        const int j = arow ? e / NB : e % NB;
        sl[j * LD + i] = v[u];
    }
    __syncthreads();
    // Column sums of |L| for ||L||_1: thread t adds 16 rows of column t % 64
    // (walked from a lane-dependent row, so that the lanes of a read fall in
    // different banks).  sp: partial sums of L, of inv(L), reciprocals.
    const int lane = t & 63, wv = t >> 6;
    auto partial_sums = [&](T *part) {
        T a = T(0);
#pragma unroll
        for (int u = 0; u < 16; ++u) a += fabs(sl[lane * LD + 16 * wv + ((u + lane) & 15)]);
        part[t] = a;
    };
    T *rinv = sp + 512;
    if (F != nullptr) partial_sums(sp);
    // 1. inverses of the 16 x 16 diagonal blocks b: lane (b, c) solves D_b y =
    // e_c.  Each of its 16 quotients is a product with the reciprocal of the
    // diagonal and one correction by the exact remainder (Markstein's step: the
    // quotient rounded, as a division gives it, in three dependent operations
    // instead of a division's dozen); a block with an entry whose reciprocal or
    // remainder could leave the normal range takes the divisions.
    T x[16];
    const int o1 = 16 * ((t & 63) >> 4), c1 = t & 15;
    T *blk16 = sl + o1 * LD + o1;
    if (t < 64) {
        const T d = sl[t * LD + t], ad = fabs(d);
        constexpr T big = Mma16<T>::big, small = T(1) / big;
        const bool plain = __all(ad >= small && ad <= big);
        rinv[t] = T(1) / d;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = (i == c1) ? T(1) : T(0);
        if (plain) {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const T dj = blk16[j * LD + j], rj = rinv[o1 + j];
                const T q = x[j] * rj;
                x[j] = fma(fma(-q, dj, x[j]), rj, q);
#pragma unroll
                for (int r = j + 1; r < 16; ++r) x[r] -= blk16[j * LD + r] * x[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                x[j] = x[j] / blk16[j * LD + j];
#pragma unroll
                for (int r = j + 1; r < 16; ++r) x[r] -= blk16[j * LD + r] * x[j];
            }
        }
    }
    __syncthreads();  // every lane has read its block, and every wave L for its column sums
    if (t < 64) {
#pragma unroll
        for (int i = 0; i < 16; ++i) blk16[c1 * LD + i] = x[i];
    }
    __syncthreads();
    // Products of 16 x 16 blocks on MFMA.  A result's registers are the right
    // operand of the next product as they stand (step s of lane l takes k =
    // kmap(l / 16, s)), so C inv(D) never goes through LDS.
    typedef Mma16<T> MM;
    typename MM::acc_t step3[2];
    const int lo = lane & 15, kk = lane >> 4;
    // acc += L(rows r0.., cols c0..) * x, or * L(rows c0.., cols d0..)
    auto left = [&](int r0, int c0, const typename MM::acc_t &x, typename MM::acc_t acc) {
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = MM::mma(sl[(c0 + MM::kmap(kk, s)) * LD + r0 + lo], x[s], acc);
        return acc;
    };
    auto both = [&](int r0, int c0, int d0, typename MM::acc_t acc) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = MM::mma(sl[(c0 + MM::kmap(kk, s)) * LD + r0 + lo], sl[(d0 + lo) * LD + c0 + MM::kmap(kk, s)], acc);
        return acc;
    };
    auto put = [&](int r0, int c0, const typename MM::acc_t &v) {
#pragma unroll
        for (int s = 0; s < 4; ++s) sl[(c0 + lo) * LD + r0 + MM::kmap(kk, s)] = -v[s];
    };
    const typename MM::acc_t zero = {T(0), T(0), T(0), T(0)};
    // 2. two 32-blocks, wave p: C_p <- -inv(D_2p+1) C_p inv(D_2p)
    if (wv < 2) {
        const int o = 32 * wv;
        const typename MM::acc_t x = both(o + 16, o, o, zero);
        put(o + 16, o, left(o + 16, o + 16, x, zero));
    }
    __syncthreads();
    // 3. the 64-block: Q <- -inv(R) Q inv(P), wave b a 16-column half of Q
    if (wv < 2) {
        const int c = 16 * wv;
        typename MM::acc_t x0 = zero, x1 = zero;
        if (wv == 0) {
            x0 = both(32, 0, 0, x0);
            x1 = both(48, 0, 0, x1);
        }
        x0 = both(32, 16, c, x0);
        x1 = both(48, 16, c, x1);
        const typename MM::acc_t y0 = left(32, 32, x0, zero);
        const typename MM::acc_t y1 = left(48, 48, x1, left(48, 32, x0, zero));
        __builtin_amdgcn_sched_barrier(0);
        step3[0] = y0;
        step3[1] = y1;
    }
    __syncthreads();  // Q read by both waves
    if (wv < 2) {
        put(32, 16 * wv, step3[0]);
        put(48, 16 * wv, step3[1]);
    }
    __syncthreads();
    // write: column-major 64 x 64; an upper block's inverse is J inv(L) J
    T *w = W + blk * NB * NB;
#pragma unroll 8
    for (int e = t; e < NB * NB; e += NT) {
        int i = e % NB, j = e / NB;  // element (i, j) of the stored inverse
        T val;
        if (lower || i >= nb || j >= nb)
            val = (i < nb && j < nb) || lower ? sl[j * LD + i] : (i == j ? T(1) : T(0));
        else
            val = sl[(nb - 1 - j) * LD + (nb - 1 - i)];
        w[e] = val;
    }
    // Condition of the block, kappa_1 = ||L||_1 ||inv(L)||_1 (both exact, the
    // inverse being in LDS): an explicitly inverted block applied as a
    // product has backward error growing with kappa * u, so a block above
    // LEAF_REFINE_KAPPA is flagged and the panels follow its product with
    // one step of refinement (X += inv(L) (B - L X)).
    if (F != nullptr) {
        partial_sums(sp + 256);
        __syncthreads();
        if (t < 64) {
            T nl = sp[t] + sp[t + 64] + sp[t + 128] + sp[t + 192];
            T ni = sp[t + 256] + sp[t + 320] + sp[t + 384] + sp[t + 448];
            for (int o = 32; o > 0; o >>= 1) {
                const T l = __shfl_xor(nl, o), i = __shfl_xor(ni, o);
                nl = l > nl ? l : nl;
                ni = i > ni ? i : ni;
            }
            if (t == 0) {
                const T kappa = nl * ni;
                F[blk] = (kappa > T(LEAF_REFINE_KAPPA) || !(kappa == kappa)) ? 1 : 0;
            }
        }
    }
}

// Inverse of one NB x NB diagonal block per work-group, by forward
// substitution on the columns of the identity (one column per lane, the
// block in LDS).  Each column of the inverse is a backward-stable triangular
// solve; the inverses turn the diagonal-block leaves of the recursion into
// MFMA products.
template <typename T, int NB>
__device__ __forceinline__ void trtri_block(int64_t n, int64_t blk, const T *__restrict__ A, int64_t rs, int64_t cs, bool lower,
                            bool unit, T *__restrict__ W, T *sl, T *srinv) {
    const int t = threadIdx.x;
    const int64_t off = blk * NB;
    const int nb = (int)(n - off < NB ? n - off : NB);
    // canonical lower L: the block itself, or J*U*J for an upper block
    const T *base = lower ? A + off * (rs + cs) : A + (off + nb - 1) * (rs + cs);
    const int64_t ars = lower ? rs : -rs, acs = lower ? cs : -cs;
    const bool arow = (ars == 1 || ars == -1);
    constexpr int SB = 16;
#pragma unroll 1
    for (int e0 = 0; e0 < NB * NB; e0 += SB * LEAF_COLS) {
        T v[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            int e = e0 + u * LEAF_COLS + t;
            int i = arow ? e % NB : e / NB;
            int j = arow ? e / NB : e % NB;
            if (e < NB * NB && i < nb && j < nb && !(unit && i == j))
                v[u] = (j <= i) ? base[i * ars + j * acs] : T(0);
            else
                v[u] = (i == j) ? T(1) : T(0);
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            int e = e0 + u * LEAF_COLS + t;
            int i = arow ? e % NB : e / NB;
            int j = arow ? e / NB : e % NB;
            if (e < NB * NB) sl[j * NB + i] = v[u];
        }
    }
    for (int i = t; i < NB; i += LEAF_COLS) srinv[i] = (i < nb && !unit) ? T(1) / base[i * ars + i * acs] : T(1);
    __syncthreads();
    if (t >= NB) return;
    T x[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) x[i] = (i == t) ? T(1) : T(0);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        x[j] = x[j] * srinv[j];
#pragma unroll
        for (int r = j + 1; r < NB; ++r) x[r] = x[r] - sl[j * NB + r] * x[j];
    }
    // column t of inv(L); for an upper block inv(U) = J inv(L) J
    T *w = W + blk * NB * NB;
    if (lower || t >= nb) {
#pragma unroll
        for (int i = 0; i < NB; ++i) w[i + t * NB] = x[i];
    } else {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            if (i < nb) w[(nb - 1 - i) + (nb - 1 - t) * NB] = x[i];
            else w[i + (nb - 1 - t) * NB] = T(0);
        }
    }
}

// Inverse of one NB x NB diagonal block per work-group, by forward
// substitution on the columns of the identity (one column per lane, the
// block in LDS).  Each column of the inverse is a backward-stable triangular
// solve; the inverses turn the diagonal-block leaves of the recursion into
// MFMA products.
template <typename T, int NB>
__global__ __launch_bounds__(LEAF_COLS) void trtri_kernel(int64_t n, const T *__restrict__ A, int64_t rs,
                                                          int64_t cs, int lower, int unit, T *__restrict__ W) {
    __shared__ __attribute__((aligned(16))) T sl[NB * NB];
    __shared__ T srinv[NB];
    trtri_block<T, NB>(n, blockIdx.x, A, rs, cs, lower != 0, unit != 0, W, sl, srinv);
}

// The 64-block inverse used by the recursion and the batched solver.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void trtri64_kernel(int64_t n, const T *__restrict__ A, int64_t rs, int64_t cs,
                                                      int lower, int unit, T *__restrict__ W, int *__restrict__ F) {
    __shared__ __attribute__((aligned(16))) T sl[64 * TRTRI_LD];
    __shared__ T sp[TRTRI_SP];
    trtri64_block<T>(n, blockIdx.x, A, rs, cs, lower != 0, unit != 0, W, sl, sp, F);
}

// Batched form: one work-group per (system, block) pair.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void batch_trtri_kernel(const BatchSys<T> *__restrict__ sys,
                                                         const int2 *__restrict__ blk) {
    __shared__ __attribute__((aligned(16))) T sl[64 * TRTRI_LD];
    __shared__ T sp[TRTRI_SP];
    const int2 b = blk[blockIdx.x];
    const BatchSys<T> &S = sys[b.x];
    // the diagonal blocks of the effective matrix in its natural orientation:
    // for a right-side system M = op(A)^T, whose blocks are the transposed
    // blocks of op(A); the inverses are stored for op(A) (read transposed).
    const bool right = (S.wrs != 1);
    const int64_t rs = right ? S.mcs : S.mrs, cs = right ? S.mrs : S.mcs;
    const bool lower = right ? (S.lower == 0) : (S.lower != 0);
    trtri64_block<T>(S.n, b.y, S.M, rs, cs, lower, false, (T *)S.W, sl, sp, (int *)S.F);
}

template <typename T>
hipError_t launch_batch_trtri(const BatchSys<T> *sys, const int2 *blk, int nblk, hipStream_t s) {
    if (nblk <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_trtri_kernel<T>, dim3(nblk), dim3(256), 0, s, sys, blk);
    return hipGetLastError();
}

template hipError_t launch_batch_trtri<float>(const BatchSys<float> *, const int2 *, int, hipStream_t);
template hipError_t launch_batch_trtri<double>(const BatchSys<double> *, const int2 *, int, hipStream_t);

template <typename T>
hipError_t launch_trtri_blocks(int64_t n, int nb, const T *A, int64_t rs, int64_t cs, bool lower, T *W,
                               hipStream_t s, bool unit, int *flags) {
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + nb - 1) / nb;
    const int lo = lower ? 1 : 0, un = unit ? 1 : 0;
    if (nb == 64)
        hipLaunchKernelGGL((trtri64_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, s, n, A, rs, cs, lo, un, W,
                           flags);
    else if (nb == 32)
        hipLaunchKernelGGL((trtri_kernel<T, 32>), dim3((unsigned)blocks), dim3(LEAF_COLS), 0, s, n, A, rs, cs, lo, un,
                           W);
    else if (nb == 16)
        hipLaunchKernelGGL((trtri_kernel<T, 16>), dim3((unsigned)blocks), dim3(LEAF_COLS), 0, s, n, A, rs, cs, lo, un,
                           W);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

template hipError_t launch_trtri_blocks<float>(int64_t, int, const float *, int64_t, int64_t, bool, float *,
                                               hipStream_t, bool, int *);
template hipError_t launch_trtri_blocks<double>(int64_t, int, const double *, int64_t, int64_t, bool, double *,
                                                hipStream_t, bool, int *);

template <typename T, int NB, bool ICONTIG>
static hipError_t launch_leaf_nb(const LeafArgs<T> &a, hipStream_t s) {
    int64_t groups = (a.m + LEAF_COLS - 1) / LEAF_COLS;
    if (a.trmm)
        hipLaunchKernelGGL((leaf_kernel<T, NB, ICONTIG, true>), dim3((unsigned)groups), dim3(LEAF_COLS), 0, s, a.nb,
                           a.m, a.A, a.ars, a.acs, a.B, a.brs, a.bcs, a.scale);
    else
        hipLaunchKernelGGL((leaf_kernel<T, NB, ICONTIG, false>), dim3((unsigned)groups), dim3(LEAF_COLS), 0, s, a.nb,
                           a.m, a.A, a.ars, a.acs, a.B, a.brs, a.bcs, a.scale);
    return hipGetLastError();
}

template <typename T, bool ICONTIG>
static hipError_t launch_leaf_stage(const LeafArgs<T> &a, hipStream_t s) {
    if (a.nb <= 16) return launch_leaf_nb<T, 16, ICONTIG>(a, s);
    if (a.nb <= 32) return launch_leaf_nb<T, 32, ICONTIG>(a, s);
    return launch_leaf_nb<T, 64, ICONTIG>(a, s);
}

template <typename T>
hipError_t launch_leaf(const LeafArgs<T> &a, hipStream_t s) {
    if (a.m <= 0 || a.nb <= 0) return hipSuccess;
    if (a.nb > LEAF_MAX_NB) return hipErrorInvalidValue;
    if (a.brs == 1 || a.brs == -1) return launch_leaf_stage<T, true>(a, s);
    return launch_leaf_stage<T, false>(a, s);
}

template hipError_t launch_leaf<float>(const LeafArgs<float> &, hipStream_t);
template hipError_t launch_leaf<double>(const LeafArgs<double> &, hipStream_t);

// Fill an m-by-n column-major block with zeros (alpha == 0 semantics of the
// BLAS: B is set to zero without being read).
template <typename T>
__global__ void zero_kernel(int64_t rows, int64_t cols, T *__restrict__ B, int64_t ldb) {
    int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t total = rows * cols;
    for (; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        int64_t i = idx % rows, j = idx / rows;
        B[i + j * ldb] = T(0);
    }
}

template <typename T>
hipError_t launch_zero(int64_t rows, int64_t cols, T *B, int64_t ldb, hipStream_t s) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    int64_t total = rows * cols;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(zero_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s, rows, cols, B, ldb);
    return hipGetLastError();
}

template hipError_t launch_zero<float>(int64_t, int64_t, float *, int64_t, hipStream_t);
template hipError_t launch_zero<double>(int64_t, int64_t, double *, int64_t, hipStream_t);

}  // namespace nla
