// Fused diagonal-panel solve: the bottom levels of the recursion in one
// launch, and the persistent batched solver built on the same routine.
//
// For a diagonal block of up to NBIG rows of the effective triangular matrix
// M (lower or upper), a work-group owns a strip of W right-hand-side columns,
// keeps that strip of B in LDS for the whole block and runs the blocked
// algorithm the recursion would run below this size:
//   TRSM lower: for k: X_k = inv(M_kk) B_k ; B_i -= M_ik X_k (i > k)
//   TRSM upper: the same from the last 64-block backwards (i < k)
//   TRMM lower: from the last block up: B_i = tri(M_ii) B_i + sum_{k<i} M_ik B_k
//   TRMM upper: from the first block down, sum over k > i
// with inv(M_kk) from the batched diagonal inverses.  Each phase is a
// 64 x W x 64 MFMA product whose M-operand fragments are fetched one phase
// ahead; no work-group depends on another (each owns its columns).
//
// Replaces the bottom of unified_rec (src/rectrxm.jl:101-198) together with the
// leaves it calls (src/trsm.jl:128-150, src/trmm.jl:332-393); the batched form
// has no counterpart in the reference (one call per system there).
#include "nla_device.h"
#include "nla_internal.h"

namespace nla {

#define NLA_LDS __attribute__((address_space(3)))

// The source of the M-operand elements outside a block (or its triangle):
// reading zeros there leaves nothing to mask when the fragment is used.
static __device__ __align__(16) const double panel_zero[2] = {0.0, 0.0};

// 16x16x4 f32 MFMA (2048 flops, 32 cycles): D[i][j] in lane j+16*(i/4),
// register i%4 (verified on gfx950 by a lane-layout probe).
struct Mfma16f {
    static constexpr int BD = 16, KD = 4, NR = 4;
    typedef f4_t acc_t;
    __device__ static inline acc_t zero() { return acc_t{0.f, 0.f, 0.f, 0.f}; }
    __device__ static inline acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static inline int di(int l, int r) { return 4 * (l >> 4) + r; }
    __device__ static inline int dj(int l, int) { return l & 15; }
};

// Output tile of one phase: 64 rows x W columns over 4 waves.  With 16x16
// MFMA blocks and W = 16, wave w owns rows 16w..16w+15 of the 64-row block;
// narrow strips give many work-groups (m/16) for the column parallelism.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> : Mfma<double> {};
template <>
struct Mfma16<float> : Mfma16f {};

template <typename T, int W_>
struct PanelShape {
    typedef Mfma16<T> MF;
    static constexpr int W = W_, CBW = W_ / 16;
    static_assert(W_ % 16 == 0, "strip width");
    __device__ static inline int rb0(int wave) { return wave; }
    __device__ static inline int cb0(int) { return 0; }
};

// A phase of the blocked algorithm for nsb 64-blocks.  kind: 0 = diagonal
// (TRSM: inv(M_kk) block; TRMM: masked M_ii), 1 = off-diagonal M_ik.
struct Phase {
    int i, k, kind;
    bool first, last;  // first / last phase of an output block group
};

// Phase (step, q) of the blocked algorithm, walked in order with phase_next
// (step s holds s + 1 phases for TRSM, nsb - s for TRMM).
__device__ inline Phase phase_at(int step, int q, int nsb, bool lower, bool trmm) {
    Phase ph;
    if (!trmm) {
        // Left-looking: output block i (top-down for lower, bottom-up for
        // upper) gathers its sources k (already solved) in registers, then
        // its diagonal phase subtracts them from B_i and applies inv(M_ii).
        // Step s has s source phases and one diagonal phase.
        const int i = lower ? step : nsb - 1 - step;
        ph.i = i;
        if (q < step) {
            ph.k = lower ? q : nsb - 1 - q;
            ph.kind = 1;
            ph.first = (q == 0);
            ph.last = false;
        } else {
            ph.k = i;
            ph.kind = 0;
            ph.first = (step == 0);
            ph.last = true;
        }
    } else {
        // output block i (bottom-up for lower): diagonal, then its sources
        const int i = lower ? nsb - 1 - step : step;
        ph.i = i;
        if (q == 0) {
            ph.k = i;
            ph.kind = 0;
        } else {
            ph.k = lower ? q - 1 : i + q;
            ph.kind = 1;
        }
        ph.first = (q == 0);
        ph.last = (q == nsb - step - 1);
    }
    return ph;
}

__device__ inline void phase_next(int &step, int &q, int nsb, bool trmm) {
    ++q;
    if (trmm ? (q >= nsb - step) : (q > step)) {
        ++step;
        q = 0;
    }
}

__device__ inline int phase_count(int nsb, bool trmm) {
    (void)trmm;
    return nsb * (nsb + 1) / 2;
}

// Solve / multiply one strip of W columns (starting at c0) of one diagonal
// panel; bs is the LDS strip (W x LDB).  Four waves: wave w computes rows
// 16w..16w+15 of every 64-row phase over its 64-deep k range.
template <typename T, int NBIG, int WS, bool TRMM>
// Always inlined: with the single-panel kernel and the batched kernel both
// calling one instantiation, the compiler otherwise emits a real call (and
// the panel ran 50 % slower).
__device__ __forceinline__ void panel_strip(int nbig, int64_t m, int64_t c0, const T *__restrict__ Mp, int64_t mrs,
                                            int64_t mcs, bool lower, bool unit, T *__restrict__ Bp, int64_t brs,
                                            int64_t bcs,
                                            const T *__restrict__ Wp, int64_t wrs, int64_t wcs, T scale,
                                            const int *__restrict__ Fp, NLA_LDS T *bs, NLA_LDS T *sc = nullptr,
                                            unsigned *xmax = nullptr) {
    typedef PanelShape<T, WS> PS;
    typedef typename PS::MF MF;
    constexpr int W = PS::W;
    constexpr int LDB = NBIG + (sizeof(T) == 8 ? 2 : 4);
    constexpr int NKS = 64 / MF::KD;  // k-steps per 64-deep phase
    constexpr int NW = 4, NT = NW * 64, NKW = NKS;

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int nsb = (nbig + 63) / 64;

    // ---- load the strip (coalesced along B's contiguous direction) ----
    // Each thread issues a batch of independent loads before it stores any
    // of them, so their latencies overlap; no division per element.
    //   rowc (unit row stride): thread t takes rows t, t+256, ... of every
    //   column; otherwise (unit column stride) it takes column t % W of rows
    //   t / W, t / W + 256 / W, ...
    const bool rowc = (brs == 1 || brs == -1);
    const int nrow = nsb * 64;  // rows past nbig up to the 64-boundary are zeroed
    static_assert(NT % W == 0, "strip width must divide the work-group");
    constexpr int RSTEP = NT / W;
    if (rowc) {
        for (int r = t; r < nrow; r += NT) {
            T v[W];
#pragma unroll
            for (int c = 0; c < W; ++c) {
                const bool ok = r < nbig && c0 + c < m;
                v[c] = *(ok ? Bp + r * brs + (c0 + c) * bcs : Bp);
                v[c] = ok ? (TRMM ? v[c] : v[c] * scale) : T(0);
            }
#pragma unroll
            for (int c = 0; c < W; ++c) bs[c * LDB + r] = v[c];
        }
    } else {
        const int c = t % W;
        const bool cok = c0 + c < m;
        constexpr int SL = 8;
        for (int r0 = t / W; r0 < nrow; r0 += RSTEP * SL) {
            T v[SL];
#pragma unroll
            for (int u = 0; u < SL; ++u) {
                const int r = r0 + u * RSTEP;
                const bool ok = cok && r < nbig;
                v[u] = *(ok ? Bp + r * brs + (c0 + c) * bcs : Bp);
                v[u] = ok ? (TRMM ? v[u] : v[u] * scale) : T(0);
            }
#pragma unroll
            for (int u = 0; u < SL; ++u) {
                const int r = r0 + u * RSTEP;
                if (r < nrow) bs[c * LDB + r] = v[u];
            }
        }
    }
    __syncthreads();

    const int lo = lane % MF::BD, lk = lane / MF::BD;
    const int rb = PS::rb0(wave), cbase = PS::cb0(wave);
    // two accumulator sets (even / odd k-steps) keep two independent MFMA
    // chains in flight per wave; they are summed when a block is written
    typename MF::acc_t acc[PS::CBW], acc2[PS::CBW];
    auto bsize = [&](int b) { return (b == nsb - 1) ? nbig - 64 * b : 64; };

    // M-operand fragment of phase ph: op(i, k) for this lane's row.  Elements
    // outside the block (or, for the TRMM diagonal, outside the triangle) are
    // read from panel_zero, so no instruction waits for the loads before the
    // fragment is used, one phase later.
    //
    // The lane's elements of a phase are op(i, kb + KD sw), sw < NKW, each
    // KD * acs past the last: one 64-bit add per load (a multiply per load
    // before, at a quarter of the rate).  Which of them lie inside the block
    // (and its triangle) is a prefix / suffix of sw, computed once per phase
    // as a bit mask.
    static_assert(MF::KD == 4, "four k per MFMA step");
    const int fi = rb * MF::BD + lo;            // the lane's row of a block
    const int kb = lk;                          // the lane's first k
    auto span = [](int c) { return c <= 0 ? 0u : (c >= NKW ? (NKW >= 32 ? ~0u : (1u << NKW) - 1u) : (1u << c) - 1u); };
    // global address space spelled out: a select between the block and
    // panel_zero otherwise degrades the loads to flat ones; its address is
    // taken once (the compiler would rebuild it before every select)
    typedef const __attribute__((address_space(1))) T GT;
    GT *zp = (GT *)panel_zero;
    asm volatile("" : "+v"(zp));
    // the lane's offset and the step between its k in M and W blocks
    const int64_t offM = (int64_t)fi * mrs + (int64_t)kb * mcs, stM = (int64_t)MF::KD * mcs;
    const int64_t offW = (int64_t)fi * wrs + (int64_t)kb * wcs, stW = (int64_t)MF::KD * wcs;
    auto fetch = [&](const Phase &ph, T *af) {
        const T *A;
        int64_t off, st;
        int tri = 0;
        if (ph.kind == 0 && !TRMM) {
            A = Wp + (int64_t)ph.k * 64 * 64;
            off = offW;
            st = stW;
        } else {
            A = Mp + (int64_t)(64 * ph.i) * mrs + (int64_t)(64 * ph.k) * mcs;
            off = offM;
            st = stM;
            if (ph.kind == 0) tri = lower ? 1 : 2;
        }
        const int ni = bsize(ph.i), nk = bsize(ph.k);
        // k < nk: the first ceil((nk - kb) / 4) steps; a unit diagonal is not
        // read (the strict triangle here, the block itself added when the
        // result is written)
        uint32_t bits = fi < ni ? span((nk - kb + 3) >> 2) : 0u;
        if (tri == 1) bits &= span((((unit ? fi - 1 : fi) - kb) >> 2) + 1);             // k <= i (k < i)
        if (tri == 2) bits &= ~span(((unit ? fi + 1 : fi) - kb + 3) >> 2);            // k >= i (k > i)
        GT *p = (GT *)(A + off);
        if (tri == 0 && ni == 64 && nk == 64) {  // a whole block (uniform): nothing to select
#pragma unroll
            for (int sw = 0; sw < NKW; ++sw) {
                af[sw] = *p;
                p += st;
            }
        } else {
#pragma unroll
            for (int sw = 0; sw < NKW; ++sw) {
                af[sw] = *(((bits >> sw) & 1u) ? p : zp);
                p += st;
            }
        }
    };
    auto compute = [&](const Phase &ph, const T *af) {
        const NLA_LDS T *src = bs + ph.k * 64;
        // all LDS operands of the phase are requested before the first MFMA
        T bv[NKW][PS::CBW];
#pragma unroll
        for (int sw = 0; sw < NKW; ++sw)
#pragma unroll
            for (int cb = 0; cb < PS::CBW; ++cb)
                bv[sw][cb] = src[((cbase + cb) * MF::BD + lo) * LDB + sw * MF::KD + lk];
        // keep the scheduler from sinking the reads back next to their MFMAs
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);  // issue priority while in the MFMA cluster
#pragma unroll
        for (int sw = 0; sw < NKW; ++sw) {
            const T a = af[sw];
#pragma unroll
            for (int cb = 0; cb < PS::CBW; ++cb) {
                if (sw & 1) acc2[cb] = MF::mma(a, bv[sw][cb], acc2[cb]);
                else acc[cb] = MF::mma(a, bv[sw][cb], acc[cb]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
    };
    auto write_block = [&](int ib, T alpha, T beta) {
        NLA_LDS T *dst = bs + ib * 64;
#pragma unroll
        for (int cb = 0; cb < PS::CBW; ++cb)
#pragma unroll
            for (int r = 0; r < MF::NR; ++r) {
                const int row = rb * MF::BD + MF::di(lane, r);
                const int col = (cbase + cb) * MF::BD + MF::dj(lane, r);
                NLA_LDS T *p = dst + col * LDB + row;
                T v = alpha * (acc[cb][r] + acc2[cb][r]);
                *p = (beta == T(0)) ? v : v + beta * *p;
            }
    };
    auto zero_acc = [&]() {
#pragma unroll
        for (int cb = 0; cb < PS::CBW; ++cb) {
            acc[cb] = MF::zero();
            acc2[cb] = MF::zero();
        }
    };
    // An ill-conditioned diagonal block (flag set by the inverse kernel):
    // X_i = inv(M_ii) B_i followed by one refinement step X_i += inv(M_ii)
    // (B_i - M_ii X_i) (backward stable while kappa(M_ii) * u << 1).  A
    // rare path, in plain FMAs: thread t owns row t % 64 of the block and
    // columns t / 64 + NW * j; X goes through the 64 x W scratch sc.
    auto solve_refined = [&](int ib) {
        constexpr int NC = W / NW;
        const int r = t & 63, cg = t >> 6;
        const int nb = bsize(ib);
        const T *Wk = Wp + (int64_t)ib * 64 * 64;
        const T *Mk = Mp + (int64_t)(64 * ib) * (mrs + mcs);
        NLA_LDS T *blk = bs + ib * 64;
        T x[NC], v[NC];
        // X = inv(M_ii) B_i (the inverse is zero outside its triangle and
        // the identity past nb)
#pragma unroll
        for (int j = 0; j < NC; ++j) x[j] = T(0);
        for (int k = 0; k < 64; ++k) {
            const T w = Wk[r * wrs + k * wcs];
#pragma unroll
            for (int j = 0; j < NC; ++j) x[j] += w * blk[(cg + NW * j) * LDB + k];
        }
#pragma unroll
        for (int j = 0; j < NC; ++j) sc[(cg + NW * j) * 64 + r] = x[j];
        __syncthreads();
        // R = B_i - M_ii X
#pragma unroll
        for (int j = 0; j < NC; ++j) v[j] = unit ? sc[(cg + NW * j) * 64 + r] : T(0);
        if (r < nb) {
            const int k0 = lower ? 0 : (unit ? r + 1 : r);
            const int k1 = lower ? (unit ? r : r + 1) : nb;
            for (int k = k0; k < k1; ++k) {
                const T a = Mk[r * mrs + k * mcs];
#pragma unroll
                for (int j = 0; j < NC; ++j) v[j] += a * sc[(cg + NW * j) * 64 + k];
            }
        }
#pragma unroll
        for (int j = 0; j < NC; ++j) v[j] = blk[(cg + NW * j) * LDB + r] - v[j];
        __syncthreads();  // every thread has read B_i
#pragma unroll
        for (int j = 0; j < NC; ++j) blk[(cg + NW * j) * LDB + r] = v[j];
        __syncthreads();
        // X += inv(M_ii) R
        for (int k = 0; k < 64; ++k) {
            const T w = Wk[r * wrs + k * wcs];
#pragma unroll
            for (int j = 0; j < NC; ++j) x[j] += w * blk[(cg + NW * j) * LDB + k];
        }
        __syncthreads();  // every thread has read R
#pragma unroll
        for (int j = 0; j < NC; ++j) blk[(cg + NW * j) * LDB + r] = x[j];
        __syncthreads();  // X_i complete for the blocks that follow
    };
    // The accumulators are zero when an output block's first phase starts:
    // cleared once here and after every write that consumes them (a
    // conditional clear in the source phases cost a select per register).
    zero_acc();
    auto run = [&](const Phase &ph, const T *af) {
        if (!TRMM) {
            if (ph.kind == 1) {  // acc += M_ik X_k, kept in registers
                compute(ph, af);
            } else {  // B_i -= acc; X_i = inv(M_ii) B_i, in place
                if (!ph.first) write_block(ph.i, T(-1), T(1));
                zero_acc();
                __syncthreads();
                if (Fp != nullptr && Fp[ph.i] != 0) {
                    solve_refined(ph.i);
                    return;
                }
                compute(ph, af);
                __syncthreads();  // every wave has read B_i
                write_block(ph.i, T(1), T(0));
                zero_acc();
                __syncthreads();  // X_i complete for the blocks that follow
            }
            return;
        }
        compute(ph, af);
        if (ph.last) {
            __syncthreads();  // every wave has read B_i
            write_block(ph.i, T(1), unit ? T(1) : T(0));
            zero_acc();
            __syncthreads();
        }
    };

    // phases with the M-operand fragments of the next PD - 1 phases in
    // flight: a ring of PD register buffers, the loop body unrolled PD
    // times so every buffer index is a compile-time constant.  Fetches are
    // unconditional (past the last phase they repeat it): a fetch under a
    // branch made the compiler wait for it at the join, before the phase
    // that did not need it.
    constexpr int PD = 2;
    const int np = phase_count(nsb, TRMM);
    T fr[PD][NKW];
    Phase phr[PD];
    // the next phase to fetch, as (step, q) and its index
    int fstep = 0, fq = 0, fp = 0;
    auto fetch_next = [&](int slot) {
        phr[slot] = phase_at(fstep, fq, nsb, lower, TRMM);
        fetch(phr[slot], fr[slot]);
        if (fp + 1 < np) {  // past the last phase, repeat it
            phase_next(fstep, fq, nsb, TRMM);
            ++fp;
        }
    };
#pragma unroll
    for (int j = 0; j < PD - 1; ++j) fetch_next(j);
    const int np_full = np - np % PD;
    for (int p = 0; p < np_full; p += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            fetch_next((u + PD - 1) % PD);
            run(phr[u], fr[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < PD - 1; ++u)
        if (np_full + u < np) run(phr[u], fr[u]);

    // ---- write the strip back ----
    T vmax = T(0);  // largest |X| written (fp32 TRSM with xmax)
    if (rowc) {
        for (int r = t; r < nbig; r += NT) {
#pragma unroll
            for (int c = 0; c < W; ++c) {
                const T v = bs[c * LDB + r];
                if (c0 + c < m) {
                    Bp[r * brs + (c0 + c) * bcs] = TRMM ? v * scale : v;
                    if (!TRMM) vmax = fabs(v) > vmax ? fabs(v) : vmax;
                }
            }
        }
    } else {
        const int c = t % W;
        if (c0 + c < m) {
            for (int r = t / W; r < nbig; r += RSTEP) {
                const T v = bs[c * LDB + r];
                Bp[r * brs + (c0 + c) * bcs] = TRMM ? v * scale : v;
                if (!TRMM) vmax = fabs(v) > vmax ? fabs(v) : vmax;
            }
        }
    }
    if constexpr (sizeof(T) == 4 && !TRMM) {
        if (xmax != nullptr) {
            // a NaN compares false above and never raises the maximum; the
            // refinement's own checks see it in the residual.  One global
            // atomic per work-group: every work-group of the launch targets
            // the same slot, and one per wave serialized there (+10 us per
            // launch).
            __shared__ unsigned s_max;
            unsigned b = __float_as_uint((float)vmax);
            for (int o = 32; o > 0; o >>= 1) {
                const unsigned u = __shfl_xor(b, o);
                b = u > b ? u : b;
            }
            if (t == 0) s_max = 0u;
            __syncthreads();
            if ((t & 63) == 0) atomicMax(&s_max, b);
            __syncthreads();
            if (t == 0 && s_max != 0u) atomicMax(xmax, s_max);
        }
    }
}

// The left-looking strip of the batched solver as one launch: for panels with
// little of a chain or more strips than compute units (below), and above 512
// rows (taken only when a larger panel size is set).
template <typename T, int NBIG, int WS, bool TRMM>
__global__ __launch_bounds__(256) void panel_left_kernel(int nbig, int64_t m, const T *__restrict__ Mp,
                                                             int64_t mrs, int64_t mcs, int lower, int unit,
                                                             T *__restrict__ Bp, int64_t brs, int64_t bcs,
                                                             const T *__restrict__ Wp, int64_t wrs, int64_t wcs,
                                                             T scale, const int *__restrict__ Fp, unsigned *xmax) {
    constexpr int LDB = NBIG + (sizeof(T) == 8 ? 2 : 4);
    __shared__ __attribute__((aligned(16))) T bs_raw[WS * LDB];
    // the refinement step's scratch
    __shared__ __attribute__((aligned(16))) T sc_raw[!TRMM ? 64 * WS : 1];
    panel_strip<T, NBIG, WS, TRMM>(nbig, m, (int64_t)blockIdx.x * WS, Mp, mrs, mcs, lower != 0, unit != 0, Bp,
                                       brs, bcs, Wp, wrs, wcs, scale, Fp, (NLA_LDS T *)bs_raw,
                                       (NLA_LDS T *)sc_raw, xmax);
}

// ---------------------------------------------------------------------------
// Panels of up to 512 rows: a work-group of eight waves per strip of W
// columns, the strip in LDS.
//
// What bounds a panel: with few strips the chain of diagonal blocks, with
// many the matrix cores, and in between the rate at which a CU's address
// unit takes load instructions (16 cycles each whatever their width: with one
// element per lane the M operand's loads took as long as its FP64 MFMAs, and
// twice as long in FP32).  So:
//   - the rows are dealt out in units of 32, two MFMA row blocks, and a lane
//     loads the two rows 2l, 2l + 1 of a column of M at once, or four
//     consecutive k where M is contiguous along k (KC);
//   - TRSM runs right-looking.  A wave owns units w and w + 8 (in solving
//     order) and keeps sum M_ik X_k of each in its accumulators, apart from
//     B as the left-looking order does, so nothing of its precision is lost;
//     a step subtracts the sums of one 64-block from B, multiplies by the
//     inverse (four waves) and then all waves add the new block's products
//     to every unit still owed at once.  Two barriers per 64-block;
//   - a 32-deep piece of M is always on its way while the one before it is
//     used.  The loops have no load under a branch (the compiler would wait
//     at the join): a wave's steps are split by which of its units are still
//     active, and the waves that apply the inverse run their own copy;
//   - TRMM has no chain: the waves form whole units from the strip in LDS, long
//     ones paired with short ones.

template <typename T>
struct Mat2 {
    typedef T v2_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    typedef T v4_t __attribute__((ext_vector_type(4), aligned(sizeof(T))));
};

constexpr int PU_WAVES = 8, PU_MAX = 512;

// One unit's rows of M: row block b of the unit holds rows 2l + b (l = lane %
// 16), or 16 b + l where M is contiguous along k.
template <typename T, bool KC>
struct PanelRows {
    const T *p[KC ? 2 : 1];  // the lane's row(s), at its k = 4 (lane / 16)
    int64_t cs;
    __device__ static inline int row(int b, int lo) { return KC ? 16 * b + lo : 2 * lo + b; }
    // r0: the unit's first row; rows past the panel read its last row (an
    // even row's pair may reach one element past it, which is the next column
    // of a matrix that has one: off the diagonal k + 1 < nbig)
    __device__ inline void init(const T *M, int64_t mrs, int64_t mcs, int r0, int nbig, int lane) {
        const int lo = lane & 15, kk = 4 * (lane >> 4);
        cs = mcs;
#pragma unroll
        for (int b = 0; b < (KC ? 2 : 1); ++b) {
            const int r = r0 + row(b, lo);
            p[b] = M + (int64_t)(r < nbig ? r : nbig - 1) * mrs + (int64_t)kk * mcs;
        }
    }
    // f[b][4 q + e] = M(row b, k0 + 16 q + kk + e), q < 2
    __device__ inline void load(int k0, T (*f)[8]) const {
        if constexpr (KC) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    if constexpr (sizeof(T) == 8) {
                        const typename Mat2<T>::v2_t x = *(const typename Mat2<T>::v2_t *)(p[b] + k0 + 16 * q);
                        const typename Mat2<T>::v2_t y = *(const typename Mat2<T>::v2_t *)(p[b] + k0 + 16 * q + 2);
                        f[b][4 * q] = x[0];
                        f[b][4 * q + 1] = x[1];
                        f[b][4 * q + 2] = y[0];
                        f[b][4 * q + 3] = y[1];
                    } else {
                        const typename Mat2<T>::v4_t x = *(const typename Mat2<T>::v4_t *)(p[b] + k0 + 16 * q);
#pragma unroll
                        for (int e = 0; e < 4; ++e) f[b][4 * q + e] = x[e];
                    }
                }
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const typename Mat2<T>::v2_t x =
                        *(const typename Mat2<T>::v2_t *)(p[0] + (int64_t)(k0 + 16 * q + e) * cs);
                    f[0][4 * q + e] = x[0];
                    f[1][4 * q + e] = x[1];
                }
        }
    }
};

// The same element by element, zero (and not read) outside [lo_k, hi_k) of
// its row: M(r, k0 + ...) with r the row block's row.
template <typename T>
__device__ __forceinline__ void panel_masked(const T *__restrict__ M, int64_t mrs, int64_t mcs, int r, int k0, int ka,
                                             int kb, int lane, T *f) {
    // global address space spelled out: a select between the block and
    // panel_zero otherwise degrades the loads to flat ones
    typedef const __attribute__((address_space(1))) T GT;
    GT *zp = (GT *)panel_zero;
    const int kk = 4 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = k0 + 16 * q + kk + e;
            f[4 * q + e] = *(k >= ka && k < kb ? (GT *)(M + (int64_t)r * mrs + (int64_t)k * mcs) : zp);
        }
}

// Sums of NB row blocks, in two sets (even and odd k of a lane): two
// independent MFMA chains, and sums half as long to round.
template <typename T, int NB, int CBW>
struct PanelAcc {
    typedef Mfma16<T> MF;
    typename MF::acc_t a[2][NB][CBW];
    __device__ inline void zero() {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int cb = 0; cb < CBW; ++cb) a[i][b][cb] = MF::zero();
    }
    __device__ inline T at(int b, int cb, int e) const { return a[0][b][cb][e] + a[1][b][cb][e]; }
};

// acc += f (32 deep) times x: xs points at the lane's column and its first k
// in LDS, column blocks 16 * ldx apart.
template <typename T, int CBW, int NB>
__device__ __forceinline__ void panel_mul(const T (*f)[8], const NLA_LDS T *xs, int ldx,
                                          PanelAcc<T, NB, CBW> &acc) {
    typedef Mfma16<T> MF;
    T x[CBW][8];
#pragma unroll
    for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[cb][4 * q + e] = xs[cb * 16 * ldx + 16 * q + e];
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc.a[e & 1][b][cb] = MF::mma(x[cb][e], f[b][e], acc.a[e & 1][b][cb]);
    __builtin_amdgcn_s_setprio(0);
}

template <typename T>
constexpr int panel_pad() {
    return 16 / (int)sizeof(T);  // 16-byte LDS reads of 16 columns start in different banks
}

// The strip between B and LDS, along B's contiguous direction, loads in
// batches so that their latencies overlap; rows past the panel and columns
// past m are zero in LDS.
template <typename T, int W, int LDB>
__device__ __forceinline__ void panel_load(const T *__restrict__ Bp, int64_t brs, int64_t bcs, int nbig, int nrow,
                                           int64_t ncol, T scale, NLA_LDS T *bs) {
    constexpr int NT = PU_WAVES * 64;
    const int t = threadIdx.x;
    if (brs == 1) {
        for (int r = t; r < nrow; r += NT) {
            T v[W];
#pragma unroll
            for (int c = 0; c < W; ++c) {
                const bool ok = r < nbig && c < ncol;
                v[c] = *(ok ? Bp + r + c * bcs : Bp);
                v[c] = ok ? v[c] * scale : T(0);
            }
#pragma unroll
            for (int c = 0; c < W; ++c) bs[c * LDB + r] = v[c];
        }
    } else {
        const int c = t % W;
        const bool cok = c < ncol;
        constexpr int SL = 8, RSTEP = NT / W;
        for (int r0 = t / W; r0 < nrow; r0 += RSTEP * SL) {
            T v[SL];
#pragma unroll
            for (int u = 0; u < SL; ++u) {
                const int r = r0 + u * RSTEP;
                const bool ok = cok && r < nbig;
                v[u] = *(ok ? Bp + r * brs + c * bcs : Bp);
                v[u] = ok ? v[u] * scale : T(0);
            }
#pragma unroll
            for (int u = 0; u < SL; ++u)
                if (r0 + u * RSTEP < nrow) bs[c * LDB + r0 + u * RSTEP] = v[u];
        }
    }
}

template <typename T, int W, int LDB>
__device__ __forceinline__ T panel_store(T *__restrict__ Bp, int64_t brs, int64_t bcs, int nbig, int64_t ncol,
                                         const NLA_LDS T *bs) {
    constexpr int NT = PU_WAVES * 64;
    const int t = threadIdx.x;
    T vmax = T(0);  // a NaN compares false and never raises it
    if (brs == 1) {
        for (int r = t; r < nbig; r += NT) {
#pragma unroll
            for (int c = 0; c < W; ++c) {
                const T v = bs[c * LDB + r];
                if (c < ncol) {
                    Bp[r + c * bcs] = v;
                    vmax = fabs(v) > vmax ? fabs(v) : vmax;
                }
            }
        }
    } else {
        const int c = t % W;
        if (c < ncol) {
            for (int r = t / W; r < nbig; r += NT / W) {
                const T v = bs[c * LDB + r];
                Bp[r * brs + c * bcs] = v;
                vmax = fabs(v) > vmax ? fabs(v) : vmax;
            }
        }
    }
    return vmax;
}

// One strip's TRSM.  bs: the strip (W x LDB), tmp: a 64 x W block.
template <typename T, int W, int LDB, bool KC>
struct PanelSolve {
    typedef Mfma16<T> MF;
    typedef PanelRows<T, KC> PR;
    static constexpr int CBW = W / 16, LDX = 64 + panel_pad<T>();
    typedef PanelAcc<T, 1, CBW> X;  // a row block of X
    int nbig, nsb, lane, wv, lo, kk;
    bool lower, unit;
    const T *Mp;
    int64_t mrs, mcs;
    const T *Wp;
    int64_t wrs, wcs;
    const int *Fp;
    NLA_LDS T *bs, *tmp;
    PR rows[2];
    PanelAcc<T, 2, CBW> acc[2];
    T fw[16];

    __device__ inline int block(int s) const { return lower ? s : nsb - 1 - s; }
    // first row of the j-th unit of this wave (in solving order)
    __device__ inline int unit_row(int j) const {
        const int u = wv + PU_WAVES * j;
        return 64 * block(u >> 1) + 32 * (u & 1);
    }
    __device__ inline void load_inverse(int s) {
        const T *p = Wp + (int64_t)block(s < nsb ? s : nsb - 1) * 64 * 64 + (16 * wv + lo) * wrs + kk * wcs;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) fw[4 * q + e] = p[(inverse_col(q, e) - kk) * wcs];
    }
    // the inverse's columns in the order of their use (this lane's of the
    // product e of block q): the diagonal block last, towards the diagonal
    __device__ inline int inverse_col(int q, int e) const {
        return 16 * ((wv + 1 + q) & 3) + (q < 3 ? kk + e : 4 * (lower ? e : 3 - e) + (kk >> 2));
    }
    __device__ inline int k_of(int s, int h) const { return 64 * block(s) + 32 * h; }

    // tmp = B_s - (the sums of unit j)
    __device__ inline void put(int j) {
        const int r0 = unit_row(j), b0 = r0 & 63;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = cb * 16 + MF::di(lane, e), i = PR::row(b, lo);
                    const T v = bs[c * LDB + r0 + i] - acc[j].at(b, cb, e);
                    tmp[c * LDX + b0 + i] = r0 + i < nbig ? v : T(0);
                }
    }
    // x (+)= the inverse's row block times tmp, in one chain with the diagonal,
    // which has the large terms, at its end: what comes after them is rounded
    // at their size (512 x 512 FP32: 8.4e-8 L-L-N and 1.29e-7 L-L-T of the
    // result in two chains of ascending k, 7.7e-8 and 8.3e-8 so).
    __device__ inline void apply_inverse(X &x) {
        T v[CBW][16];
#pragma unroll
        for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[cb][4 * q + e] = tmp[(cb * 16 + lo) * LDX + inverse_col(q, e)];
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
            for (int cb = 0; cb < CBW; ++cb) x.a[0][0][cb] = MF::mma(v[cb][e], fw[e], x.a[0][0][cb]);
    }
    __device__ inline void put_x(int s, const X &x) {
        const int r0 = 64 * block(s) + 16 * wv + lo;
#pragma unroll
        for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                bs[(cb * 16 + MF::di(lane, e)) * LDB + r0] = r0 < nbig ? x.at(0, cb, e) : T(0);
    }
    // An ill-conditioned diagonal block: X += inv(M_ss) (B_s - M_ss X).  The
    // correction has sums of its own: the two sets that hold X may be far
    // larger than X, and would round what is added to them at their size.
    // Every wave passes the barriers.
    template <bool DIAG>
    __device__ inline void refine(int s, X &x) {
        const int bl = block(s), nb = bl == nsb - 1 ? nbig - 64 * bl : 64, i = 16 * wv + lo, r = 64 * bl + i;
        T x0[CBW][4];
        if (DIAG) put_x(s, x);
        __syncthreads();  // X complete, and every wave's product with B_s done
        if (DIAG) {
            X v;
            v.zero();
            const int ka = lower ? 0 : (unit ? i + 1 : i), kb = i < nb ? (lower ? (unit ? i : i + 1) : nb) : 0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                T g[1][8];
                panel_masked<T>(Mp, mrs, mcs, i < nb ? r : nbig - 1, 64 * bl + 32 * h, 64 * bl + ka, 64 * bl + kb, lane,
                                g[0]);
                panel_mul<T, CBW, 1>(g, bs + lo * LDB + 64 * bl + 32 * h + kk, LDB, v);
            }
#pragma unroll
            for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    NLA_LDS T *p = tmp + (cb * 16 + MF::di(lane, e)) * LDX + i;  // this lane's own element of B_s
                    x0[cb][e] = x.at(0, cb, e);
                    const T mx = unit ? v.at(0, cb, e) + x0[cb][e] : v.at(0, cb, e);
                    *p = i < nb ? *p - mx : T(0);
                }
        }
        __syncthreads();
        if (DIAG) {
            x.zero();
            apply_inverse(x);
#pragma unroll
            for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
                for (int e = 0; e < 4; ++e) x.a[0][0][cb][e] = x0[cb][e] + x.at(0, cb, e), x.a[1][0][cb][e] = T(0);
        }
    }
    // Solves block s into the strip: sums out, inverse, X in; two barriers.
    template <bool DIAG>
    __device__ inline void diagonal(int s) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (((wv + PU_WAVES * j) >> 1) == s) put(j);
        __syncthreads();
        X x;
        if (DIAG) {
            x.zero();
            apply_inverse(x);
        }
        if (Fp != nullptr && Fp[block(s)] != 0) refine<DIAG>(s, x);
        if (DIAG) put_x(s, x);
        __syncthreads();
        if (DIAG) load_inverse(s + 1);
    }
    // Steps [s0, s1) with units 0 and / or 1 of this wave still owed.
    template <bool DIAG, bool U0, bool U1>
    __device__ inline void steps(int s0, int s1) {
        if (s0 >= s1) return;
        T f[2][2][8];
        constexpr int J = U0 ? 0 : 1;
        if constexpr (U0 || U1) {
            rows[J].load(k_of(s0, 0), f[0]);
            rows[J].load(k_of(s0, 1), f[1]);
        }
        for (int s = s0; s < s1; ++s) {
            diagonal<DIAG>(s);
            const int sn = s + 1 < s1 ? s + 1 : s;  // past the last step, this block again
            const NLA_LDS T *xs = bs + lo * LDB + k_of(s, 0) + kk;
            if constexpr (U0 || U1) {
                panel_mul<T, CBW, 2>(f[0], xs, LDB, acc[J]);
                rows[U0 && U1 ? 1 : J].load(k_of(U0 && U1 ? s : sn, 0), f[0]);
                panel_mul<T, CBW, 2>(f[1], xs + 32, LDB, acc[J]);
                rows[U0 && U1 ? 1 : J].load(k_of(U0 && U1 ? s : sn, 1), f[1]);
            }
            if constexpr (U0 && U1) {
                panel_mul<T, CBW, 2>(f[0], xs, LDB, acc[1]);
                rows[0].load(k_of(sn, 0), f[0]);
                panel_mul<T, CBW, 2>(f[1], xs + 32, LDB, acc[1]);
                rows[0].load(k_of(sn, 1), f[1]);
            }
        }
    }
    // The first step of an upper panel whose last block is short: its k range
    // ends inside a 64-block.
    template <bool DIAG>
    __device__ inline void short_step() {
        diagonal<DIAG>(0);
        const int k0 = 64 * (nsb - 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int u = wv + PU_WAVES * j;
            if (u < 2 || u >= 2 * nsb) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                T f[2][8];
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    panel_masked<T>(Mp, mrs, mcs, unit_row(j) + PR::row(b, lo), k0 + 32 * h, 0, nbig, lane, f[b]);
                panel_mul<T, CBW, 2>(f, bs + lo * LDB + k0 + 32 * h + kk, LDB, acc[j]);
            }
        }
    }
    template <bool DIAG>
    __device__ inline void run() {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (wv + PU_WAVES * j < 2 * nsb) rows[j].init(Mp, mrs, mcs, unit_row(j), nbig, lane);
            else rows[j].init(Mp, mrs, mcs, 0, nbig, lane);
            acc[j].zero();
        }
        if (DIAG) load_inverse(0);
        int s = 0;
        if (!lower && (nbig & 63) != 0) {
            short_step<DIAG>();
            s = 1;
        }
        const int n0 = wv < 2 * nsb ? wv >> 1 : 0, n1 = wv + PU_WAVES < 2 * nsb ? (wv + PU_WAVES) >> 1 : 0;
        auto later = [&](int n) { return n > s ? n : s; };
        if (n1 > 0) {
            steps<DIAG, true, true>(s, n0);
            s = later(n0);
            steps<DIAG, false, true>(s, n1);
            s = later(n1);
        } else {
            steps<DIAG, true, false>(s, n0);
            s = later(n0);
        }
        steps<DIAG, false, false>(s, nsb);
        __syncthreads();
    }
};

template <typename T, int NBIG, int W, bool KC>
__device__ __forceinline__ void panel_trmm(int nbig, int64_t m, int64_t c0, const T *__restrict__ Mp, int64_t mrs,
                                           int64_t mcs, bool lower, bool unit, T *__restrict__ Bp, int64_t brs,
                                           int64_t bcs, T scale, NLA_LDS T *bs) {
    typedef Mfma16<T> MF;
    typedef PanelRows<T, KC> PR;
    constexpr int CBW = W / 16, LDB = NBIG + panel_pad<T>(), PD = 3;
    const int t = threadIdx.x, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lo = lane & 15, kk = 4 * (lane >> 4);
    const int64_t ncol = m - c0 < W ? m - c0 : W;
    T *B = Bp + c0 * bcs;
    panel_load<T, W, LDB>(B, brs, bcs, nbig, (nbig + 31) / 32 * 32, ncol, T(1), bs);
    __syncthreads();
    const int nu = (nbig + 31) / 32;
    const NLA_LDS T *xb = bs + lo * LDB + kk;
    for (int j = 0; j < 2; ++j) {
        // a unit each for the longest ones, and the shortest for the waves with
        // the shortest of those: by length, units nu - 1 - w and nu - 16 + w,
        // from the panel's top down (512 rows, 64 columns: 5 % slower upwards)
        const int q = (j == 1) == lower ? nu - 1 - wv : nu - 2 * PU_WAVES + wv, u = lower ? q : nu - 1 - q;
        if (q < 0) continue;
        const int r0 = 32 * u;
        PanelAcc<T, 2, CBW> acc;
        acc.zero();
        T sum[2][CBW][4] = {};
        // off the diagonal, whole 32-deep pieces: [ka, kb); an upper unit's last one may be short
        const int ka = lower ? 0 : r0 + 32, kb = lower ? r0 : nbig, np = (kb - ka) / 32;
        PR rows;
        rows.init(Mp, mrs, mcs, r0, nbig, lane);
        T f[PD][2][8], d[2][8];
        if (np > 0) {
#pragma unroll
            for (int v = 0; v < PD - 1; ++v) rows.load(ka + 32 * (v < np ? v : np - 1), f[v]);
        }
        // the diagonal piece, masked to the triangle (what a whole piece reads
        // beside it is dropped, whatever it holds)
        const bool whole = r0 + 32 <= nbig;
        if (whole) rows.load(r0, d);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int r = r0 + PR::row(b, lo);
            const int k0 = lower ? r0 : (unit ? r + 1 : r), k1 = lower ? (unit ? r : r + 1) : nbig;
            if (!whole) {
                panel_masked<T>(Mp, mrs, mcs, r < nbig ? r : nbig - 1, r0, k0, r < nbig ? k1 : 0, lane, d[b]);
            } else {
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int k = r0 + 16 * q + kk + e;
                        d[b][4 * q + e] = k >= k0 && k < k1 ? d[b][4 * q + e] : T(0);
                    }
            }
        }
        panel_mul<T, CBW, 2>(d, xb + r0, LDB, acc);
        if (np > 0) {
            int i = 0;
            for (; i + PD <= np; i += PD) {
#pragma unroll
                for (int v = 0; v < PD; ++v) {
                    const int nx = i + v + PD - 1;
                    rows.load(ka + 32 * (nx < np ? nx : np - 1), f[(v + PD - 1) % PD]);
                    panel_mul<T, CBW, 2>(f[v], xb + ka + 32 * (i + v), LDB, acc);
                }
                // sums of 96 products at a time: one chain along 512 rows
                // would round more than the 256-row panels and their updates
                // (FP32 R-U-N n = 4096: 3.0e-7 of the result against 2.1e-7)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum[b][cb][e] += acc.at(b, cb, e);
                acc.zero();
            }
#pragma unroll
            for (int v = 0; v < PD - 1; ++v)
                if (i + v < np) panel_mul<T, CBW, 2>(f[v], xb + ka + 32 * (i + v), LDB, acc);
        }
        if (ka + 32 * np < kb && np >= 0 && ka < kb) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
                panel_masked<T>(Mp, mrs, mcs, r0 + PR::row(b, lo), ka + 32 * np, 0, nbig, lane, d[b]);
            panel_mul<T, CBW, 2>(d, xb + ka + 32 * np, LDB, acc);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int r = r0 + PR::row(b, lo);
#pragma unroll
            for (int cb = 0; cb < CBW; ++cb)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = cb * 16 + MF::di(lane, e);
                    if (r < nbig && c < ncol) {
                        const T x = sum[b][cb][e] + acc.at(b, cb, e), v = unit ? x + bs[c * LDB + r] : x;
                        B[r * brs + c * bcs] = v * scale;
                    }
                }
        }
    }
}

template <typename T, int NBIG, int W, bool TRMM, bool KC>
__global__ __launch_bounds__(PU_WAVES * 64) void panel_kernel(int nbig, int64_t m, const T *__restrict__ Mp,
                                                              int64_t mrs, int64_t mcs, int lower, int unit,
                                                              T *__restrict__ Bp, int64_t brs, int64_t bcs,
                                                              const T *__restrict__ Wp, int64_t wrs, int64_t wcs,
                                                              T scale, const int *__restrict__ Fp, unsigned *xmax) {
    constexpr int LDB = NBIG + panel_pad<T>(), LDX = 64 + panel_pad<T>();
    __shared__ __attribute__((aligned(16))) T strip[W * LDB];
    const int64_t c0 = (int64_t)blockIdx.x * W;
    if constexpr (TRMM) {
        panel_trmm<T, NBIG, W, KC>(nbig, m, c0, Mp, mrs, mcs, lower != 0, unit != 0, Bp, brs, bcs, scale,
                                   (NLA_LDS T *)strip);
    } else {
        __shared__ __attribute__((aligned(16))) T block[W * LDX];
        const int64_t ncol = m - c0 < W ? m - c0 : W;
        const int t = threadIdx.x;
        PanelSolve<T, W, LDB, KC> P;
        P.nbig = nbig;
        P.nsb = (nbig + 63) / 64;
        P.lane = t & 63;
        P.wv = __builtin_amdgcn_readfirstlane(t >> 6);
        P.lo = P.lane & 15;
        P.kk = 4 * (P.lane >> 4);
        P.lower = lower != 0;
        P.unit = unit != 0;
        P.Mp = Mp;
        P.mrs = mrs;
        P.mcs = mcs;
        P.Wp = Wp;
        P.wrs = wrs;
        P.wcs = wcs;
        P.Fp = Fp;
        P.bs = (NLA_LDS T *)strip;
        P.tmp = (NLA_LDS T *)block;
        T *B = Bp + c0 * bcs;
        panel_load<T, W, LDB>(B, brs, bcs, nbig, 64 * P.nsb, ncol, scale, P.bs);
        __syncthreads();
        if (P.wv < 4) P.template run<true>();
        else P.template run<false>();
        const T vmax = panel_store<T, W, LDB>(B, brs, bcs, nbig, ncol, P.bs);
        if constexpr (sizeof(T) == 4) {
            if (xmax != nullptr) {
                // one global atomic per work-group: every work-group of the
                // launch targets the same slot, and one per wave serialized
                // there (+10 us per launch)
                __shared__ unsigned s_max;
                unsigned b = __float_as_uint((float)vmax);
                for (int o = 32; o > 0; o >>= 1) {
                    const unsigned u = __shfl_xor(b, o);
                    b = u > b ? u : b;
                }
                if (t == 0) s_max = 0u;
                __syncthreads();
                if ((t & 63) == 0) atomicMax(&s_max, b);
                __syncthreads();
                if (t == 0 && s_max != 0u) atomicMax(xmax, s_max);
            }
        }
    }
}

template <typename T, int NBIG, int W, bool KC>
static hipError_t launch_panel_k(const PanelArgs<T> &a, hipStream_t s) {
    const dim3 grid((unsigned)((a.m + W - 1) / W)), block(PU_WAVES * 64);
    const int lo = a.lower ? 1 : 0, un = a.unit ? 1 : 0;
    if (a.trmm)
        hipLaunchKernelGGL((panel_kernel<T, NBIG, W, true, KC>), grid, block, 0, s, a.nbig, a.m, a.M, a.mrs, a.mcs,
                           lo, un, a.B, a.brs, a.bcs, a.W, a.wrs, a.wcs, a.scale, (const int *)nullptr,
                           (unsigned *)nullptr);
    else
        hipLaunchKernelGGL((panel_kernel<T, NBIG, W, false, KC>), grid, block, 0, s, a.nbig, a.m, a.M, a.mrs, a.mcs,
                           lo, un, a.B, a.brs, a.bcs, a.W, a.wrs, a.wcs, a.scale, a.F, a.xmax);
    return hipGetLastError();
}

// The strip's LDS is sized for 128, 256 or 512 rows.
template <typename T, int W>
static hipError_t launch_panel_w(const PanelArgs<T> &a, hipStream_t s) {
    const bool kc = a.mcs == 1;
    if (a.nbig <= 128) return kc ? launch_panel_k<T, 128, W, true>(a, s) : launch_panel_k<T, 128, W, false>(a, s);
    if (a.nbig <= 256) return kc ? launch_panel_k<T, 256, W, true>(a, s) : launch_panel_k<T, 256, W, false>(a, s);
    return kc ? launch_panel_k<T, 512, W, true>(a, s) : launch_panel_k<T, 512, W, false>(a, s);
}

template <typename T, int NBIG, int WS, bool TRMM>
static hipError_t launch_panel_left(const PanelArgs<T> &a, hipStream_t s) {
    hipLaunchKernelGGL((panel_left_kernel<T, NBIG, WS, TRMM>), dim3((unsigned)((a.m + WS - 1) / WS)), dim3(256), 0, s,
                       a.nbig, a.m, a.M, a.mrs, a.mcs, a.lower ? 1 : 0, a.unit ? 1 : 0, a.B, a.brs, a.bcs, a.W, a.wrs,
                       a.wcs, a.scale, TRMM ? nullptr : a.F, TRMM ? nullptr : a.xmax);
    return hipGetLastError();
}

// 32 columns only where the setting asks for them; above 512 rows FP64's do not
// fit LDS.
template <typename T, bool TRMM>
static hipError_t launch_panel_left_n(const PanelArgs<T> &a, hipStream_t s) {
    if (a.strip == 32) {
        if (a.nbig <= 512) return launch_panel_left<T, 512, 32, TRMM>(a, s);
        if constexpr (sizeof(T) == 4) return launch_panel_left<T, 1024, 32, TRMM>(a, s);
    }
    if (a.nbig <= 128) return launch_panel_left<T, 128, 16, TRMM>(a, s);
    if (a.nbig <= 256) return launch_panel_left<T, 256, 16, TRMM>(a, s);
    if (a.nbig <= 512) return launch_panel_left<T, 512, 16, TRMM>(a, s);
    return launch_panel_left<T, 1024, 16, TRMM>(a, s);
}

// Right-hand sides per group of the eight-wave panel, or 0 for the
// left-looking strip (16 of them).  kc: M contiguous along k; bcol: B's
// contiguous direction runs along the right-hand sides; n x n panel, m of them.
//
// An eight-wave group has a CU to itself.  32 columns halve the reads of M and
// fill the matrix cores better, but a round of such groups is 8192 columns, so
// they win where they leave less than half of the last round idle (full).  Four
// waves and 16 columns leave room for two and more groups on a CU: the
// left-looking strip wins where there is little of a chain to shorten, or, for
// TRSM, more strips than CUs to hide it, but it loads M along k (kc) one
// element per cache line.  It also rounds more (TRSM of an upper M twice as
// much, TRMM above 192 rows 1.2 to 1.6 times), so of two that take about as
// long the eight waves are taken.  Within 1 % of the fastest of the three on
// average over 64 .. 512 rows and 16 .. 24000 columns.  Measured on MI355X (us,
// left / eight waves of 16 / of 32 columns, TRSM with its inverses):
//   FP64 TRSM  L-L-T 128 rows, 10000 columns 29.0 / 37.8 / 73.9; 144 rows 38.5 / 48.6 / 84.7;
//              512 rows, 8192 131 / 105 / 110; R-U-N 149 / 120 / 113; L-L-N 81.6 / 86.0 / 103
//   FP64 TRMM  L-L-N 128 rows, 10000 16.8 / 20.2 / 34.8; 320 rows 50.1 / 42.0 / 60.0;
//              L-L-T 256 rows, 8192 42.5 / 32.7 / 25.4; 10000 57.7 / 43.2 / 43.5
//   FP32 TRSM  L-L-T 512 rows, 8192 119 / 62.4 / 54.5; 10000 167 / 81.6 / 91.5; R-U-N 211 / 122 / 99.9
//   FP32 TRMM  L-L-N 144 rows, 10000 18.3 / 13.5 / 24.5; R-U-N 512 rows, 8192 126 / 50.2 / 37.9
// (32 columns for all past 4096: up to 1.9 times as long as what it replaced).
template <typename T>
static int panel_columns(bool trmm, bool kc, bool bcol, bool unit, int n, int64_t m) {
    constexpr bool F64 = sizeof(T) == 8;
    // few columns.  A unit diagonal is LU's: its blocks are as often flagged
    // for refinement as not, which the eight waves do on MFMA (64 rows 25 / 8
    // us, 128 rows 48 / 15)
    if (m <= 16 * 256) return n > 128 || (trmm ? !(F64 && kc && bcol) : unit) ? 16 : 0;
    const bool full = (m - 1) % (32 * 256) >= 16 * 256;
    if (n <= 64) return 0;
    if (!trmm) {
        if (!F64 && bcol && full) return 32;
        if (!kc || n <= 128) return 0;
        if (F64) return bcol && n > 384 && full ? 32 : 16;
        return bcol || (n > 256 && full) ? 32 : 16;
    }
    if (F64) {
        if (n <= 128 || (!kc && n <= 192 && m > 32 * 256)) return 0;
        return full || (kc && n > 384) ? 32 : 16;
    }
    if (bcol) return full ? 32 : (!kc && n <= 128 ? 0 : 16);
    return n > 320 && full ? 32 : 16;
}

template <typename T>
hipError_t launch_panel(const PanelArgs<T> &a, hipStream_t s) {
    if (a.m <= 0 || a.nbig <= 0) return hipSuccess;
    if (a.nbig > PANEL_MAX) return hipErrorInvalidValue;
    if (a.strip != 16 && a.strip != 32) return hipErrorInvalidValue;
    const int columns = a.strip == 32 ? 32 : panel_columns<T>(a.trmm, a.mcs == 1, a.brs != 1, a.unit, a.nbig, a.m);
    if (a.nbig > PU_MAX || a.waves == 4 || (a.waves == 0 && columns == 0))
        return a.trmm ? launch_panel_left_n<T, true>(a, s) : launch_panel_left_n<T, false>(a, s);
    return columns == 32 ? launch_panel_w<T, 32>(a, s) : launch_panel_w<T, 16>(a, s);
}

template hipError_t launch_panel<float>(const PanelArgs<float> &, hipStream_t);
template hipError_t launch_panel<double>(const PanelArgs<double> &, hipStream_t);

// ---------------------------------------------------------------------------
// Persistent batched solver: work-groups pull (system, strip) tasks from a
// queue ordered by decreasing cost until it is empty.  Every system is one
// diagonal panel of up to NBIG rows; the kernel is instantiated per size
// class (NBIG = 128 ... 1024) so that the LDS strip, and with it the number
// of work-groups a CU holds, fits the largest system of the class.

template <typename T, bool TRMM, int NBIG>
__global__ __launch_bounds__(256) void batch_kernel(const BatchSys<T> *__restrict__ sys,
                                                    const BatchTask *__restrict__ tasks, int ntasks,
                                                    int *__restrict__ counter) {
    constexpr int WS = BatchStrip<T>::W;
    constexpr int LDB = NBIG + (sizeof(T) == 8 ? 2 : 4);
    __shared__ __attribute__((aligned(16))) T bs_raw[WS * LDB];
    __shared__ __attribute__((aligned(16))) T sc_raw[TRMM ? 1 : 64 * WS];  // refinement scratch
    __shared__ int s_idx;
    for (;;) {
        if (threadIdx.x == 0) s_idx = atomicAdd(counter, 1);
        __syncthreads();
        const int idx = s_idx;
        __syncthreads();
        if (idx >= ntasks) break;  // every wave of the group sees the same idx
        const BatchTask tk = tasks[idx];
        const BatchSys<T> &S = sys[tk.sys];
        panel_strip<T, NBIG, WS, TRMM>(S.n, S.m, (int64_t)tk.strip * WS, S.M, S.mrs, S.mcs, S.lower != 0, false, S.B,
                                       S.brs, S.bcs, S.W, S.wrs, S.wcs, S.scale, TRMM ? nullptr : S.F,
                                       (NLA_LDS T *)bs_raw, (NLA_LDS T *)sc_raw);
        __syncthreads();
    }
}

__global__ void zero_int_kernel(int *p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}

template <typename T, bool TRMM>
static const void *batch_ptr_t(int nbig) {
    switch (nbig) {
        case 128: return (const void *)batch_kernel<T, TRMM, 128>;
        case 256: return (const void *)batch_kernel<T, TRMM, 256>;
        case 512: return (const void *)batch_kernel<T, TRMM, 512>;
        case 1024: return (const void *)batch_kernel<T, TRMM, 1024>;
        default: return nullptr;
    }
}

template <typename T>
const void *batch_kernel_ptr(bool trmm, int nbig) {
    return trmm ? batch_ptr_t<T, true>(nbig) : batch_ptr_t<T, false>(nbig);
}

template <typename T>
hipError_t launch_batch(const BatchSys<T> *sys, const BatchTask *tasks, int ntasks, int *counter, bool trmm,
                        int nbig, int groups, hipStream_t s) {
    if (ntasks <= 0) return hipSuccess;
    const void *k = batch_kernel_ptr<T>(trmm, nbig);
    if (!k) return hipErrorInvalidValue;
    hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(64), 0, s, counter);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    void *args[] = {(void *)&sys, (void *)&tasks, (void *)&ntasks, (void *)&counter};
    return hipLaunchKernel(k, dim3(groups), dim3(256), args, 0, s);
}

template const void *batch_kernel_ptr<float>(bool, int);
template const void *batch_kernel_ptr<double>(bool, int);

template hipError_t launch_batch<float>(const BatchSys<float> *, const BatchTask *, int, int *, bool, int, int,
                                        hipStream_t);
template hipError_t launch_batch<double>(const BatchSys<double> *, const BatchTask *, int, int *, bool, int, int,
                                         hipStream_t);

}  // namespace nla
