// One tile of C = beta*C + alpha*op(X)*op(Y) on gfx950 MFMA, shared by the
// GEMM update and the grouped GEMM of the batched solver.
//
// Orientation: the MFMA computes D = C^T for each 16x16 (f64) / 32x32 (f32)
// block, so that the lane index of D's column walks down a column of C and the
// epilogue writes whole 128-byte segments of the column-major output.
//
// LDS layout per operand follows its contiguous dimension in HBM:
//   outer-contiguous (X 'N', Y 'T'):   tile[k][outer]   (row stride BO + PO)
//   k-contiguous     (X 'T', Y 'N'):   tile[outer][k]   (row stride BK + PK)
// so HBM reads are 16-byte vectors along the contiguous dimension and LDS
// writes are vectors too; the transpose happens in the per-lane MFMA operand
// read instead.  Global memory takes 16-byte loads at any element's address,
// so leading dimensions need no alignment.
#pragma once

#include "nla_device.h"

namespace nla {

// Pointers into LDS keep their address space so that every access compiles
// to ds_read / ds_write (a generic pointer becomes a flat access, which also
// waits on outstanding global loads).
#define NLA_LDS __attribute__((address_space(3)))

// EDGE: the tile may reach past the operand's last outer index (no).  What
// lies past it only feeds results that are not stored, so load() clamps whole
// chunks into the operand, zeroes nothing, and lets a chunk that straddles
// the end run on into the next k (memory of the operand while VW and more k
// remain: the caller takes the last steps with load_tail()).  load_tail()
// checks every element and zeroes what is past K, in both operands: no 0 * NaN.
template <typename T, int BO, int BK, int NT, bool KCONTIG, bool EDGE>
struct TileLoader {
    // Each thread moves CH chunks of VW consecutive elements along the
    // contiguous dimension of the operand.
    static constexpr int VW = 16 / sizeof(T);
    static constexpr int CHUNKS = BO * BK / VW;
    static constexpr int CH = CHUNKS / NT;
    static_assert(CHUNKS % NT == 0, "tile does not divide among threads");
    static constexpr int PO = (sizeof(T) == 8) ? 2 : 4;  // pads keep 16-byte alignment
    static constexpr int PK = (sizeof(T) == 8) ? 2 : 4;
    static constexpr int LDS_ELEMS = KCONTIG ? BO * (BK + PK) : BK * (BO + PO);
    typedef T gvec_t __attribute__((ext_vector_type(VW), aligned(sizeof(T))));
    typedef T lvec_t __attribute__((ext_vector_type(VW)));

    T r[CH][VW];
    const T *p[CH];  // the chunks' addresses at the first step
    int last[EDGE && !KCONTIG ? CH : 1];  // the chunk's last element inside the operand
    int64_t ks;
    uint32_t okbits;   // load_tail: bit (c*VW+e) set when the element's k is in range

    // Coordinates (outer, k) inside the tile of chunk c of thread t.
    __device__ static inline void coords(int t, int c, int &o, int &k) {
        int q = t + c * NT;
        if (KCONTIG) {
            k = (q % (BK / VW)) * VW;
            o = q / (BK / VW);
        } else {
            o = (q % (BO / VW)) * VW;
            k = q / (BO / VW);
        }
    }

    // Element (outer, k) of the operand lives at P[outer*so + k*sk] with one
    // of so/sk equal to 1.  o0/k0: tile origin; no: outer extent.
    __device__ inline void init(const T *__restrict__ P, int64_t so, int64_t sk, int64_t o0, int64_t k0, int64_t no,
                                int t) {
        ks = sk;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            int o, k;
            coords(t, c, o, k);
            int64_t go = o0 + o;
            if constexpr (EDGE && KCONTIG) go = go < no ? go : no - 1;
            if constexpr (EDGE && !KCONTIG) {
                if (go >= no) go = no - 1;
                last[c] = no - 1 - go < VW - 1 ? (int)(no - 1 - go) : VW - 1;
            }
            p[c] = P + go * so + (k0 + k) * sk;
        }
    }
    // Step kt (uniform: its offset is added in scalar registers).
    __device__ inline void load(int kt) {
        const int64_t off = (int64_t)kt * BK * ks;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const gvec_t v = *reinterpret_cast<const gvec_t *>(p[c] + off);
#pragma unroll
            for (int e = 0; e < VW; ++e) r[c][e] = v[e];
        }
    }
    // Step kt, of which nk (1 .. BK) k remain; an element past them reads its
    // outer index's first k of the step.
    __device__ inline void load_tail(int kt, int nk, int t) {
        const int64_t off = (int64_t)kt * BK * ks;
        okbits = 0;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            int o, k;
            coords(t, c, o, k);
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const bool ok = (KCONTIG ? k + e : k) < nk;
                const T *q = p[c] + off;
                if constexpr (KCONTIG) r[c][e] = q[ok ? e : -k];
                else r[c][e] = (ok ? q : q - (int64_t)k * ks)[EDGE && e > last[c] ? last[c] : e];
                okbits |= (ok ? 1u : 0u) << (c * VW + e);
            }
        }
    }
    // Zero what load_tail read past K, just before the LDS store.
    __device__ inline void apply_bounds() {
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int e = 0; e < VW; ++e)
                if (!((okbits >> (c * VW + e)) & 1u)) r[c][e] = T(0);
    }

    // Zero the elements outside a triangle: keep (outer, k) when
    // (KEEP_LE ? k <= outer : k >= outer), in global coordinates.
    template <bool KEEP_LE>
    __device__ inline void mask(int64_t o0, int64_t k0, int t) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            int o, k;
            coords(t, c, o, k);
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                int64_t eo = o0 + (KCONTIG ? o : o + e);
                int64_t ek = k0 + (KCONTIG ? k + e : k);
                bool keep = KEEP_LE ? (ek <= eo) : (ek >= eo);
                if (!keep) r[c][e] = T(0);
            }
        }
    }

    __device__ inline void store(NLA_LDS T *lds, int t) const {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            int o, k;
            coords(t, c, o, k);
            NLA_LDS T *q = KCONTIG ? lds + o * (BK + PK) + k : lds + k * (BO + PO) + o;
            lvec_t v;
#pragma unroll
            for (int e = 0; e < VW; ++e) v[e] = r[c][e];
            *reinterpret_cast<NLA_LDS lvec_t *>(q) = v;
        }
    }

    // Operand element (outer, k) from the staged tile.
    __device__ static inline T at(const NLA_LDS T *lds, int o, int k) {
        return KCONTIG ? lds[o * (BK + PK) + k] : lds[k * (BO + PO) + o];
    }
};

// LDS elements of both stages of a tile's operands.
template <typename T, int BM, int BN, int BK, int WM, int WN, bool TX, bool TY>
struct TileLds {
    static constexpr int X = 2 * TileLoader<T, BM, BK, WM * WN * 64, TX, false>::LDS_ELEMS;
    static constexpr int Y = 2 * TileLoader<T, BN, BK, WM * WN * 64, !TY, false>::LDS_ELEMS;
};

// Hardware dispatches work-group g to XCD g % 8.  Renumber so each XCD owns
// a contiguous range of logical tiles, then walk tiles in groups of GM row
// tiles so the tiles resident on one XCD share X row panels and Y column
// panels in that XCD's L2.
__device__ inline void tile_coords(int G, int g, int tiles_m, int &tm, int &tn) {
    const int NX = 8, GM = 8;
    int xcd = g % NX, idx = g / NX;
    int per = G / NX, rem = G % NX;
    int gp = (xcd < rem) ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
    int tiles_n = G / tiles_m;
    int group = GM * tiles_n;
    int gid = gp / group;
    int first = gid * GM;
    int gm = tiles_m - first < GM ? tiles_m - first : GM;
    int in = gp % group;
    tm = first + in % gm;
    tn = in / gm;
}

// One BM x BN tile of C at (row0, col0).  EDGE: the tile may reach past M or
// N.  TRI: triangle mask (GemmArgs::tri).
template <typename T, int BM, int BN, int BK, int WM, int WN, bool TX, bool TY, int TRI, bool EDGE>
__device__ __forceinline__ void gemm_tile(int64_t M, int64_t N, int64_t K, T alpha, const T *__restrict__ X,
                                          int64_t ldx, const T *__restrict__ Y, int64_t ldy, T beta, T *C,
                                          int64_t ldc, int64_t row0, int64_t col0, NLA_LDS T *lds_xb,
                                          NLA_LDS T *lds_yb) {
    typedef Mfma<T> MF;
    constexpr int NT = WM * WN * 64;
    constexpr int TWM = BM / WM, TWN = BN / WN;
    constexpr int RB = TWM / MF::BD, CB = TWN / MF::BD;
    static_assert(RB >= 1 && CB >= 1 && TWM % MF::BD == 0 && TWN % MF::BD == 0, "bad wave tile");
    static_assert(BK % MF::KD == 0, "bad BK");
    // X tile: outer = rows of C, contiguous along k when TX.
    typedef TileLoader<T, BM, BK, NT, TX, EDGE> LX;
    // Y tile: outer = columns of C, contiguous along k when !TY.
    typedef TileLoader<T, BN, BK, NT, !TY, EDGE> LY;
    NLA_LDS T *lds_x[2] = {lds_xb, lds_xb + LX::LDS_ELEMS};
    NLA_LDS T *lds_y[2] = {lds_yb, lds_yb + LY::LDS_ELEMS};

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wm = wave % WM, wn = wave / WM;

    typename MF::acc_t acc[CB][RB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[cb][rb] = MF::zero();

    // k-steps that the triangle zeroes entirely are skipped: the operand's
    // rows (columns) of this tile only reach k up to (from) the tile edge.
    int64_t kbeg = 0, kend = K;
    if (TRI == 1) kend = row0 + BM < K ? row0 + BM : K;
    if (TRI == 2) kbeg = row0 < K ? row0 : K;
    if (TRI == 3) kbeg = col0 < K ? col0 : K;
    if (TRI == 4) kend = col0 + BN < K ? col0 + BN : K;
    const int64_t kn = kend - kbeg, whole = EDGE ? kn - LX::VW : kn;
    const int nfull = whole > 0 ? (int)(whole / BK) : 0, nkt = (int)((kn + BK - 1) / BK);

    LX lx;
    LY ly;
    // op(X)(r, k): TX ? X[k + r*ldx] : X[r + k*ldx];  op(Y)(k, c): TY ?
    // Y[c + k*ldy] : Y[k + c*ldy]
    lx.init(X, TX ? ldx : 1, TX ? 1 : ldx, row0, kbeg, M, t);
    ly.init(Y, TY ? 1 : ldy, TY ? ldy : 1, col0, kbeg, N, t);
    // op(X)(r,k): outer r, inner k.  op(Y)(k,c): outer c, inner k; the Y
    // triangle conditions are c <= k (lower) / c >= k (upper).  Only steps
    // that meet the diagonal need a mask.
    auto stage = [&](int kt, int buf) {
        const int64_t k0 = kbeg + (int64_t)kt * BK;
        if (TRI == 1 && k0 + BK > row0) lx.template mask<true>(row0, k0, t);
        if (TRI == 2 && k0 < row0 + BM) lx.template mask<false>(row0, k0, t);
        if (TRI == 3 && k0 < col0 + BN) ly.template mask<false>(col0, k0, t);
        if (TRI == 4 && k0 + BK > col0) ly.template mask<true>(col0, k0, t);
        lx.store(lds_x[buf], t);
        __builtin_amdgcn_sched_barrier(0);  // the stores in the order of the loads: each waits for its own
        ly.store(lds_y[buf], t);
    };
    const int lo = lane % MF::BD, lk = lane / MF::BD;
    // One k step from one stage of LDS, and a part of one: the operands of a
    // single depth into registers, and their products.
    constexpr int KS = BK / MF::KD;
    auto read = [&](int buf, int ks, T *a, T *b) {
        const NLA_LDS T *sx = lds_x[buf];
        const NLA_LDS T *sy = lds_y[buf];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) a[cb] = LY::at(sy, wn * TWN + cb * MF::BD + lo, ks * MF::KD + lk);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) b[rb] = LX::at(sx, wm * TWM + rb * MF::BD + lo, ks * MF::KD + lk);
    };
    auto products = [&](const T *a, const T *b) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) acc[cb][rb] = MF::mma(a[cb], b[rb], acc[cb][rb]);
    };
    T a[2][CB], b[2][RB];
    auto multiply = [&](int buf) {
        __builtin_amdgcn_s_setprio(1);  // issue priority to waves in their MFMA cluster
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            T a[CB], b[RB];
            read(buf, ks, a, b);
            products(a, b);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // Whole steps.  The waves of a work-group reach the end of a step together,
    // so what stands there idles the matrix cores: with the LDS stores, the
    // barrier and the first LDS reads in a row that was 4 to 8 % of the FP64
    // loop.  So the operands of a depth are read ahead of the products before
    // it, the next step's stores stand among the products (its loads were
    // issued a whole step before), and the barrier comes before the last
    // products, which cover the next step's first reads.  Measured on MI355X
    // (us, before / after): FP64 4096 x 8192 x 4096 4128 / 4016, 2048 x 2048 x
    // 1024 151 / 143, 3000^3 1217 / 1158; FP32 1531 x 1023 x 976 44.1 / 43.0.
    // Sixteen waves (FP32 256 x 256) have 128 registers each, too few for two
    // sets of operands (2023 / 2273 at 4096 x 8192 x 4096), and keep the plain
    // order.
    if constexpr (NT > 512) {
        if (nfull > 0) {
            lx.load(0);
            ly.load(0);
            stage(0, 0);
        }
        __syncthreads();
        for (int kt = 0; kt < nfull; ++kt) {
            const int cur = kt & 1;
            const bool more = kt + 1 < nfull;
            if (more) {
                lx.load(kt + 1);
                ly.load(kt + 1);
            }
            multiply(cur);
            if (more) stage(kt + 1, cur ^ 1);
            __syncthreads();
        }
    } else {
        static_assert(KS % 2 == 0, "every step starts with the same set");
        auto ahead = [&](int of) {
            __builtin_amdgcn_s_setprio(1);
            products(a[of], b[of]);
            __builtin_amdgcn_s_setprio(0);
        };
        if (nfull > 0) {
            lx.load(0);
            ly.load(0);
            stage(0, 0);
            lx.load(nfull > 1 ? 1 : 0);
            ly.load(nfull > 1 ? 1 : 0);
            __syncthreads();
            read(0, 0, a[0], b[0]);
            for (int kt = 0; kt + 1 < nfull; ++kt) {
                const int cur = kt & 1;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int to = (ks + 1) & 1;
                    if (ks + 1 < KS) {
                        read(cur, ks + 1, a[to], b[to]);
                    } else {
                        __syncthreads();
                        read(cur ^ 1, 0, a[to], b[to]);
                    }
                    ahead(ks & 1);
                    if (ks == KS - 2) {
                        stage(kt + 1, cur ^ 1);
                        const int next = kt + 2 < nfull ? kt + 2 : nfull - 1;
                        lx.load(next);
                        ly.load(next);
                    }
                }
            }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int to = (ks + 1) & 1;
                if (ks + 1 < KS) read((nfull - 1) & 1, ks + 1, a[to], b[to]);
                ahead(ks & 1);
            }
        }
        __syncthreads();
    }
    // the checked ones (at most two), on their own: a choice of loads inside
    // the loop above made the compiler wait for them before the products
    for (int kt = nfull; kt < nkt; ++kt) {
        const int64_t left = kn - (int64_t)kt * BK;
        lx.load_tail(kt, left < BK ? (int)left : BK, t);
        ly.load_tail(kt, left < BK ? (int)left : BK, t);
        lx.apply_bounds();
        ly.apply_bounds();
        stage(kt, kt & 1);
        __syncthreads();
        if constexpr (NT > 512) {
            multiply(kt & 1);
        } else {  // as in the loop: with multiply() here its registers fell worse (4032 / 4076 us at the first size)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                read(kt & 1, ks, a[0], b[0]);
                __builtin_amdgcn_s_setprio(1);
                products(a[0], b[0]);
                __builtin_amdgcn_s_setprio(0);
            }
        }
        __syncthreads();
    }

    // Epilogue: D[i][j] of block (cb, rb) is C(row j, column i).  beta is
    // uniform, so the choice is made once; with beta != 0 the C values of one
    // column block are all requested before any is used.
    if (beta == T(0)) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int r = 0; r < MF::NR; ++r) {
                    int64_t row = row0 + wm * TWM + rb * MF::BD + MF::dj(lane, r);
                    int64_t col = col0 + wn * TWN + cb * MF::BD + MF::di(lane, r);
                    if (!EDGE || (row < M && col < N)) C[row + col * ldc] = alpha * acc[cb][rb][r];
                }
    } else {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            T cv[RB][MF::NR];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int r = 0; r < MF::NR; ++r) {
                    int64_t row = row0 + wm * TWM + rb * MF::BD + MF::dj(lane, r);
                    int64_t col = col0 + wn * TWN + cb * MF::BD + MF::di(lane, r);
                    bool ok = !EDGE || (row < M && col < N);
                    cv[rb][r] = *(ok ? C + row + col * ldc : C);
                }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int r = 0; r < MF::NR; ++r) {
                    int64_t row = row0 + wm * TWM + rb * MF::BD + MF::dj(lane, r);
                    int64_t col = col0 + wn * TWN + cb * MF::BD + MF::di(lane, r);
                    if (!EDGE || (row < M && col < N))
                        C[row + col * ldc] = alpha * acc[cb][rb][r] + beta * cv[rb][r];
                }
        }
    }
}

}  // namespace nla
