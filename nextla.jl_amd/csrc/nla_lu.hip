// Recursive LU factorization with partial pivoting (nla_getrf2 in
// include/nla.h): getrf2! of the reference (src/lu.jl:185-300, LAPACK
// dgetrf2's recursion) on the device, built on this library's unit-lower
// TRSM and GEMM update.
//
// The host walks the same recursion as the reference: split the columns at
// n1 = min(m, n) / 2 (rounded up to whole panels), factor the left block, apply its row interchanges to
// the right block, solve A12 = L11^-1 A12 (unit lower), update
// A22 -= A21 A12, factor A22 and apply its interchanges to the left block.
// Panels of up to 64 columns are one kernel (the same eliminations with
// rank-1 updates in place of the GEMMs of that width), held in registers by
// work-groups that exchange one pivot row per column and take at most a
// quarter of the chip (fewer columns above 16,384 rows, in FP32 32,768; past
// 131,072 rows 8 columns in global memory).  Pivots are kept as global rows throughout (the reference shifts
// them by n1 after each recursive call).  Everything is enqueued on the
// caller's stream; pivots and info stay on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <limits>
#include <memory>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../include/nla.h"
#include "nla_internal.h"

namespace nla {

int32_t report_hip(hipError_t e, const char *where);
int32_t report_bad_arg(int k, const char *what);

namespace {

constexpr int PIV_THREADS = 1024;

// Leaf of up to LEAF_COLS columns, one work-group: for each column j the
// pivot search (src/lu.jl:223-253: first index of the largest |a|, as
// idamax), the row interchange across the leaf's columns, the scaling of the
// column below the pivot (by the reciprocal; a division below the smallest
// normal number) and the rank-1 update of the leaf's remaining columns (what
// the recursion's GEMM updates do at this width).  m == 1 is the reference's
// row case (src/lu.jl:216-221).  Pivots are written 1-based with the leaf's
// row offset r0 added (its rows start on the diagonal, r0 = its first
// column); info takes the first zero pivot's global column.  Used for blocks
// that the register panels do not take (up to LEAF_COLS columns) and to redo
// a panel (up to LEAF_COLS_MAX) whose groups did not meet.
constexpr int LEAF_COLS = 8, LEAF_COLS_MAX = 64;
constexpr int LEAF_WAVES = PIV_THREADS / 64;

// (|a|, signed a, row) of the larger |a|, ties to the smaller row.
template <typename T>
__device__ inline void better(T &bv, T &bs, int64_t &bi, T v, T sv, int64_t i) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bs = sv;
        bi = i;
    }
}

template <typename T>
__device__ inline void wave_argmax(T &bv, T &bs, int64_t &bi) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const T v = __shfl_xor(bv, o, 64), sv = __shfl_xor(bs, o, 64);
        const int64_t i = __shfl_xor(bi, o, 64);
        better(bv, bs, bi, v, sv, i);
    }
}

template <typename T>
__device__ __forceinline__ void lu_leaf_body(int64_t m, int n, T *__restrict__ A, int64_t lda, int64_t *__restrict__ ipiv,
                             int64_t *__restrict__ info, int64_t r0) {
    __shared__ T s_val[2][LEAF_WAVES], s_sgn[2][LEAF_WAVES];
    __shared__ int64_t s_row[2][LEAF_WAVES];
    __shared__ T s_u[LEAF_COLS_MAX];  // row j of the leaf after the interchange
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int kmax = (int)(m < n ? m : n);
    // partial maxima of column 0 (each later column's are taken in the
    // update pass of the column before it); the two LDS buffers alternate
    // between consecutive columns
    T bv = T(-1), bs = T(0);
    int64_t bi = m;
    for (int64_t i = t; i < m; i += PIV_THREADS) {
        const T a = A[i];
        better(bv, bs, bi, (T)fabs(a), a, i);
    }
    for (int j = 0; j < kmax; ++j) {
        const int buf = j & 1;
        T *cj = A + (int64_t)j * lda;
        wave_argmax(bv, bs, bi);
        if (lane == 0) {
            s_val[buf][wv] = bv;
            s_sgn[buf][wv] = bs;
            s_row[buf][wv] = bi;
        }
        __syncthreads();
        T pv = T(-1), a = T(0);
        int64_t p = m;
#pragma unroll
        for (int w = 0; w < LEAF_WAVES; ++w) better(pv, a, p, s_val[buf][w], s_sgn[buf][w], s_row[buf][w]);
        if (p >= m) {  // no finite maximum (all NaN): keep row j
            p = j;
            a = cj[j];
        }
        if (t == 0) {
            ipiv[j] = r0 + p + 1;
            if (a == T(0) && *info == 0) *info = r0 + j + 1;
        }
        // interchange rows j and p of the leaf's columns; row j's new values
        // go to LDS for the update
        if (t < n) {
            T *ct = A + (int64_t)t * lda;
            const T xj = ct[j], xp = ct[p];
            if (a != T(0) && p != j) {
                ct[j] = xp;
                ct[p] = xj;
                s_u[t] = xp;
            } else {
                s_u[t] = xj;
            }
        }
        __syncthreads();
        bv = T(-1);
        bs = T(0);
        bi = m;
        if (a != T(0)) {
            // scale column j below the pivot, update the columns to its right
            // and take the partial maxima of column j + 1.  Rows go in chunks
            // of RU per thread and columns in chunks of NC; every load of a
            // chunk is issued before its first store, with addresses clamped
            // to row / column j and results masked.
            constexpr int RU = 4, NC = LEAF_COLS - 1;
            const bool recip = fabs(a) >= std::numeric_limits<T>::min();
            const T r = T(1) / a;
            for (int64_t i0 = j + 1 + t; i0 < m; i0 += RU * PIV_THREADS) {
                T l[RU], x[NC][RU];
#pragma unroll
                for (int u = 0; u < RU; ++u) {
                    const int64_t i = i0 + (int64_t)u * PIV_THREADS;
                    l[u] = cj[i < m ? i : j];
                }
#pragma unroll
                for (int u = 0; u < RU; ++u) {
                    const int64_t i = i0 + (int64_t)u * PIV_THREADS;
                    l[u] = recip ? l[u] * r : l[u] / a;
                    if (i < m) cj[i] = l[u];
                }
                for (int c0 = j + 1; c0 < n; c0 += NC) {
#pragma unroll
                    for (int q = 0; q < NC; ++q) {
                        const T *cc = A + (int64_t)(c0 + q < n ? c0 + q : j) * lda;
#pragma unroll
                        for (int u = 0; u < RU; ++u) {
                            const int64_t i = i0 + (int64_t)u * PIV_THREADS;
                            x[q][u] = cc[i < m ? i : j];
                        }
                    }
#pragma unroll
                    for (int q = 0; q < NC; ++q) {
                        const int c = c0 + q;
                        if (c >= n) break;
                        T *cc = A + (int64_t)c * lda;
                        const T uc = s_u[c];
#pragma unroll
                        for (int u = 0; u < RU; ++u) {
                            const int64_t i = i0 + (int64_t)u * PIV_THREADS;
                            if (i < m) {
                                const T y = x[q][u] - l[u] * uc;
                                cc[i] = y;
                                if (c == j + 1) better(bv, bs, bi, (T)fabs(y), y, i);
                            }
                        }
                    }
                }
            }
        } else if (j + 1 < kmax) {
            // a zero column (the max |a| is 0): nothing to eliminate
            T *cn = A + (int64_t)(j + 1) * lda;
            for (int64_t i = j + 1 + t; i < m; i += PIV_THREADS) {
                const T x = cn[i];
                better(bv, bs, bi, (T)fabs(x), x, i);
            }
        }
        // no barrier here: the next column's first barrier follows every
        // thread's updates, and s_u is rewritten only after it
    }
}

template <typename T>
__global__ __launch_bounds__(PIV_THREADS) void lu_leaf_kernel(int64_t m, int n, T *__restrict__ A, int64_t lda,
                                                              int64_t *__restrict__ ipiv, int64_t *__restrict__ info,
                                                              int64_t r0) {
    lu_leaf_body<T>(m, n, A, lda, ipiv, info, r0);
}

// The same leaf for up to REG_ROWS rows, held in registers from the first load
// to the final store: one work-group, two barriers per column and nothing in
// memory in between.  Its columns cost more with the rows (REG_RPT of them per
// thread), those of the panel of several groups below do not, but that one has
// a longer start and a recovery launch behind it: a call of few columns and
// rows is faster here (narrow(), in LuRec).
constexpr int REG_THREADS = 512, REG_RPT = 8, REG_ROWS = REG_THREADS * REG_RPT;

template <typename T>
__global__ __launch_bounds__(REG_THREADS) void lu_leaf_reg_kernel(int m, int n, T *__restrict__ A, int64_t lda,
                                                                  int64_t *__restrict__ ipiv,
                                                                  int64_t *__restrict__ info, int64_t r0) {
    constexpr int W = REG_THREADS / 64;
    __shared__ T s_val[W], s_sgn[W];
    __shared__ int64_t s_row[W];
    __shared__ T s_u[LEAF_COLS], s_o[LEAF_COLS];  // the pivot row, row j before the interchange
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int kmax = m < n ? m : n;
    T a[REG_RPT][LEAF_COLS];
#pragma unroll
    for (int r = 0; r < REG_RPT; ++r) {
        const int i = t + r * REG_THREADS;
#pragma unroll
        for (int c = 0; c < LEAF_COLS; ++c) a[r][c] = (i < m && c < n) ? A[i + (int64_t)c * lda] : T(0);
    }
#pragma unroll
    for (int j = 0; j < LEAF_COLS; ++j) {
        if (j >= kmax) break;
        T bv = T(-1), bs = T(0);
        int64_t bi = m;
#pragma unroll
        for (int r = 0; r < REG_RPT; ++r) {
            const int i = t + r * REG_THREADS;
            if (i >= j && i < m) better(bv, bs, bi, (T)fabs(a[r][j]), a[r][j], (int64_t)i);
        }
        wave_argmax(bv, bs, bi);
        if (lane == 0) {
            s_val[wv] = bv;
            s_sgn[wv] = bs;
            s_row[wv] = bi;
        }
        __syncthreads();
        T pv = T(-1), av = T(0);
        int64_t p = m;
#pragma unroll
        for (int w = 0; w < W; ++w) better(pv, av, p, s_val[w], s_sgn[w], s_row[w]);
        const bool none = p >= m;  // no finite maximum (all NaN): keep row j
        if (none) p = j;
#pragma unroll
        for (int r = 0; r < REG_RPT; ++r) {
            const int i = t + r * REG_THREADS;
            if (i == p) {
#pragma unroll
                for (int c = 0; c < LEAF_COLS; ++c) s_u[c] = a[r][c];
            }
            if (i == j) {
#pragma unroll
                for (int c = 0; c < LEAF_COLS; ++c) s_o[c] = a[r][c];
            }
        }
        __syncthreads();
        if (none) av = s_o[j];
        if (t == 0) {
            ipiv[j] = r0 + p + 1;
            if (av == T(0) && *info == 0) *info = r0 + j + 1;
        }
        if (av != T(0)) {
            const bool swap = p != j, recip = fabs(av) >= std::numeric_limits<T>::min();
            const T rc = T(1) / av;
#pragma unroll
            for (int r = 0; r < REG_RPT; ++r) {
                const int i = t + r * REG_THREADS;
                if (swap && i == j) {
#pragma unroll
                    for (int c = 0; c < LEAF_COLS; ++c) a[r][c] = s_u[c];
                } else if (swap && i == p) {
#pragma unroll
                    for (int c = 0; c < LEAF_COLS; ++c) a[r][c] = s_o[c];
                }
                if (i > j && i < m) {
                    const T l = recip ? a[r][j] * rc : a[r][j] / av;
                    a[r][j] = l;
#pragma unroll
                    for (int c = j + 1; c < LEAF_COLS; ++c) a[r][c] = a[r][c] - l * s_u[c];
                }
            }
        }
        // s_val is rewritten before the next column's first barrier, s_u after
        // it: both were last read before one
    }
#pragma unroll
    for (int r = 0; r < REG_RPT; ++r) {
        const int i = t + r * REG_THREADS;
        if (i < m) {
#pragma unroll
            for (int c = 0; c < LEAF_COLS; ++c)
                if (c < n) A[i + (int64_t)c * lda] = a[r][c];
        }
    }
}

// The same factorization of a panel of up to NB columns, held in registers
// by G work-groups of NT threads with R rows per thread from the first load
// to the final store.  What bounds it is the chain of columns, not the
// arithmetic, so a column is two trips through memory (the candidates, the
// winner's row) and two work-group barriers, with everything that the next
// candidate does not need moved off that chain:
//   1. after the pivot row arrives, a thread first forms its entry of the
//      next column; each wave reduces its candidate (the largest |a| among
//      its live rows, ties to the smaller position) on DPP moves and wave 0
//      publishes the group's;
//   2. only then are the other columns updated, and the wave that holds the
//      group's candidate publishes that row and the reciprocal of its pivot,
//      while the candidates travel;
//   3. wave 0 reads all candidates and then the winner's row.  A 64-bit word
//      carries 32 bits of payload under a 32-bit tag that names the launch
//      and the column, so a reader polls the data itself: no counter, no
//      fence.  The slots alternate with the column's parity: a group
//      publishes column j + 2 only after all groups have published j + 1,
//      which each does after its last read of column j.
// The register columns move down by one with the update itself
// (a[c] = a[c + 1] - l u[c + 1]), so the column loop stays rolled and the
// kernel small; the finished column of L goes to LDS.  Rows are not moved: a
// row keeps its thread and carries its position, and is stored to its final
// position at the end.
//
// Measured on MI355X, FP64: 166 us per 64 columns at 1,000 to 8,192 rows
// (2.6 us per column: about 2 us in the two trips, whatever the number of
// groups), 73 us in one group up to 128 rows; 8-column leaves with a counter
// per column took 480 us above 4,096 rows and 256 us below, plus the
// launches between them.  Groups of 64, 128 and 256 rows measure alike; all
// groups on one XCD, with agent- or L2-scope words, is no faster.
//
// The groups of a panel wait for each other, so they must all get a place.  At
// most LU_MAX_WG are launched, on at most 64 CUs (LU_CUS: the rows of one group
// times its columns fill half of a CU's LDS, or a whole one's with 64 groups):
// a process runs four kernels at a time unless it asks for more hardware
// queues, so four LUs on streams of their own, of any height, hold the chip
// together instead of keeping parts of it from each other.  A cooperative
// launch would guarantee a place, but costs about 150 us once other streams
// have been used.  Each wait is bounded, so a group that is not resident
// (another persistent grid holds the CUs) cannot hang the others.  Every group
// saves its rows before its first exchange (and group 0 the prior info), and a
// wait that runs out raises a flag; the one-work-group recovery launch that
// follows every such panel returns at once unless the flag is up, and
// otherwise restores the saved block and factors it with the global-memory
// leaf, so the factorization stays exact.
// A single group (ONE) exchanges nothing: one barrier per column.
constexpr int LU_MAX_WG = 128;              // groups of one panel (two polled per lane)
constexpr int LU_CUS = 64;                  // compute units that a panel may hold: a quarter of the chip
constexpr int SYNC_EPOCH = 0, SYNC_LEAVE = 1;
// words 2, 3 of the buffer: the timeout flag and the info value saved before
// the panel; then, for both parities, the groups' candidates (three arrays of
// one word per group, so that a poll of all of them touches few lines) and
// their rows; then the saved block (column c at c * m)
constexpr int SYNC_FLAG = 2, SYNC_INFO = 3;
constexpr int SYNC_SLOTS = 64, HEAD_WORDS = 3 * LU_MAX_WG, ROW_WORDS = 136;
constexpr int PAR_WORDS = HEAD_WORDS + LU_MAX_WG * ROW_WORDS;
constexpr int SYNC_WORDS = SYNC_SLOTS + 2 * PAR_WORDS;
// rows of a 64-column panel: half the columns for twice as many, and so on
template <typename T>
constexpr int64_t PANEL_M_MAX = sizeof(T) == 8 ? 64 * 256 : 128 * 256;
constexpr int64_t PANEL_M_ALL = 131072;  // rows of any panel
constexpr int64_t SAVE_BYTES = PANEL_M_MAX<double> * 64 * 8;
static_assert(PANEL_M_MAX<double> * 8 == PANEL_M_MAX<float> * 4, "one buffer serves both types");
constexpr int64_t SPLIT_SPIN_LIMIT = int64_t(1) << 20;  // about a second of polling

__device__ inline void st_agent(uint64_t *p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline uint64_t ld_agent(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Columns of the register panel for m rows, 0 where the panel does not take them.
template <typename T>
inline int panel_cols(int64_t m) {
    int nb = 64;
    for (int64_t most = PANEL_M_MAX<T>; m > most && nb > 8; most *= 2) nb /= 2;
    return m <= PANEL_M_ALL ? nb : 0;
}

__device__ __forceinline__ double lane_double(double v, int l) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, l);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// The wave's largest v (no NaN; lanes without a row hold -2) and the
// smallest position that has it; returns its lane.  Six DPP steps instead
// of shuffles through LDS; several lanes with the same value are rare (a
// zero column), so their positions are compared one by one.
__device__ __forceinline__ int wave_best(double v, int pos, double &best, int &bpos) {
    double x = v;
#define NLA_DPP_MAX(CTRL)                                                                                   \
    {                                                                                                       \
        const uint64_t b = (uint64_t)__double_as_longlong(x), id = (uint64_t)__double_as_longlong(-2.0);    \
        const unsigned lo = __builtin_amdgcn_update_dpp((int)id, (int)b, CTRL, 0xf, 0xf, false);            \
        const unsigned hi = __builtin_amdgcn_update_dpp((int)(id >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false); \
        x = fmax(x, __longlong_as_double((long long)(((uint64_t)hi << 32) | lo)));                          \
    }
    NLA_DPP_MAX(0x111)  // row_shr 1, 2, 4, 8
    NLA_DPP_MAX(0x112)
    NLA_DPP_MAX(0x114)
    NLA_DPP_MAX(0x118)
    NLA_DPP_MAX(0x142)  // row_bcast 15, 31
    NLA_DPP_MAX(0x143)
#undef NLA_DPP_MAX
    best = lane_double(x, 63);
    uint64_t who = best > -2.0 ? __ballot(v == best) : 1;  // a wave without rows: lane 0's position (none)
    int l = __ffsll((unsigned long long)who) - 1;
    bpos = __builtin_amdgcn_readlane(pos, l);
    for (who &= who - 1; who; who &= who - 1) {
        const int l2 = __ffsll((unsigned long long)who) - 1;
        const int p2 = __builtin_amdgcn_readlane(pos, l2);
        if (p2 < bpos) {
            bpos = p2;
            l = l2;
        }
    }
    return l;
}

template <typename T, int NB, int R, int NT, bool ONE>
__global__ __launch_bounds__(NT) void lu_panel_kernel(int m, int n, T *__restrict__ A, int64_t lda,
                                                      int64_t *__restrict__ ipiv, int64_t *__restrict__ info,
                                                      int64_t r0, uint64_t *__restrict__ sync, int64_t spin_limit) {
    constexpr int W = NT / 64, ROWS = NT * R;
    static_assert(NB == 8 || (NB <= 64 && NB % 16 == 0), "a wave publishes one row");
    __shared__ T s_l[NB][ROWS];                                       // finished columns (and rows of U)
    __shared__ __attribute__((aligned(16))) T s_row[2][W][NB + 2];    // each wave's candidate row, entry c at c + 1
    __shared__ __attribute__((aligned(16))) T s_u[2][NB + 2];         // the pivot row, entry c at c + 1; 1 / pivot at 0
    __shared__ double s_v[2][W];
    __shared__ int s_pos[2][W], s_src[2][W];
    __shared__ int s_p[2], s_own[2], s_fail;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int G = (int)gridDim.x, g = (int)blockIdx.x;
    const int first = g * ROWS;
    const int kmax = m < n ? m : n;
    T a[R][NB];
    int pos[R];  // the row's position; -1 - position once it is a pivot row (or past m)
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = first + t + r * NT;
#pragma unroll
        for (int c = 0; c < NB; ++c) a[r][c] = (i < m && c < n) ? A[i + (int64_t)c * lda] : T(0);
        pos[r] = i < m ? i : -1 - i;
    }
    if (t == 0) s_fail = 0;
    unsigned epoch = 0;
    if constexpr (!ONE) {
        // the block as it was, for the recovery launch
        T *save = reinterpret_cast<T *>(sync + SYNC_WORDS);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (pos[r] >= 0) {
#pragma unroll
                for (int c = 0; c < NB; ++c)
                    if (c < n) save[pos[r] + (int64_t)c * m] = a[r][c];
            }
        }
        if (g == 0 && t == 0) st_agent(sync + SYNC_INFO, (uint64_t)*info);
        epoch = (unsigned)ld_agent(sync + SYNC_EPOCH);
    }
    // The group's candidate of column j from the threads' entries x of it:
    // (|pivot|, position, wave, LDS row); one barrier.  br: the candidate's
    // row of this thread, wl: this wave's candidate lane.
    double gv;
    int gp, gw, gs, br, wl;
    auto candidate = [&](int j, const T *x, auto write_row) {
        const int par = j & 1;
        double bv = -2.0;
        int bp = 0x7fffffff;
        br = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            double v = fabs((double)x[r]);
            v = v >= 0.0 ? v : -1.0;  // a NaN only wins where there is nothing else: the first live row stays
            v = pos[r] >= 0 ? v : -2.0;
            if (v > bv || (R > 1 && v == bv && pos[r] >= 0 && pos[r] < bp)) {
                bv = v;
                bp = pos[r];
                br = r;
            }
        }
        double wbest;
        int wpos;
        wl = wave_best(bv, bp, wbest, wpos);
        if (lane == wl) {
            s_v[par][wv] = wbest;
            s_pos[par][wv] = wpos;
            s_src[par][wv] = t + br * NT;
            write_row();
        }
        __syncthreads();
        gv = s_v[par][0];
        gp = s_pos[par][0];
        gs = s_src[par][0];
        gw = 0;
#pragma unroll
        for (int w = 1; w < W; ++w) {
            const double v = s_v[par][w];
            const int q = s_pos[par][w], sr = s_src[par][w];
            if (v > gv || (v == gv && v > -2.0 && q < gp)) {
                gv = v;
                gp = q;
                gs = sr;
                gw = w;
            }
        }
    };
    // this thread's candidate row (entry c at c + 1), by its lane
    auto put_row = [&](T *dst, auto width) {
        constexpr int WD = decltype(width)::value;
#pragma unroll
        for (int c = 0; c < WD; ++c) {
            T x = a[0][c];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                T y = a[r][c];
                asm("" : "+v"(y));  // a select of values: one of addresses would put the rows in memory
                if (br == r) x = y;
            }
            dst[c + 1] = x;
        }
    };
    // Column j eliminated with pivot row u (position p, LDS row src of this
    // group if own).  Each thread's entry of column j + 1 comes first
    // (next()), then the other columns.
    auto eliminate = [&](int j, int p, bool own, int src, const T *u, bool have_rc, auto width, auto next) {
        constexpr int WD = decltype(width)::value;
        const T av = u[1];
        if (g == 0 && t == 0) {
            ipiv[j] = r0 + p + 1;
            if (av == T(0) && *info == 0) *info = r0 + j + 1;
        }
        T x[R];
        if (av != T(0)) {
            // the pivot row is row j of U from here on
            if (own && wv == W - 1 && lane < WD && j + lane < NB) s_l[j + lane][src] = u[lane + 1];
            const bool recip = fabs(av) >= std::numeric_limits<T>::min();
            const T rc = have_rc ? u[0] : T(1) / av, u1 = u[2];
            T l[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (pos[r] == p) pos[r] = -1 - j;
                else if (pos[r] == j) pos[r] = p;
                l[r] = recip ? a[r][0] * rc : a[r][0] / av;
                x[r] = a[r][1] - l[r] * u1;
            }
            next(x);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (pos[r] >= 0) s_l[j][t + r * NT] = l[r];
                a[r][0] = x[r];
            }
#pragma unroll
            for (int c = 1; c + 1 < WD; ++c) {
                const T uc = u[c + 2];
#pragma unroll
                for (int r = 0; r < R; ++r) a[r][c] = a[r][c + 1] - l[r] * uc;
            }
        } else {
            // nothing to eliminate and nothing moved: the row at position j is
            // row j of U as it stands
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (pos[r] == j) {
                    pos[r] = -1 - j;
#pragma unroll
                    for (int c = 0; c < WD; ++c)
                        if (j + c < NB) s_l[j + c][t + r * NT] = a[r][c];
                } else if (pos[r] >= 0) {
                    s_l[j][t + r * NT] = a[r][0];
                }
                x[r] = a[r][1];
            }
            next(x);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c + 1 < WD; ++c) a[r][c] = a[r][c + 1];
        }
    };
    // One group: column j from its own candidate; WD: register columns still
    // in use (the panel's last columns run with narrower copies of the code).
    auto column_one = [&](int j, auto width) {
        const int par = j & 1;
        T x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = a[r][0];
        candidate(j, x, [&] { put_row(s_row[par][wv], width); });
        eliminate(j, gp, true, gs, s_row[par][gw], false, width, [](const T *) {});
    };
    uint64_t *heads = nullptr, *rows = nullptr;
    uint64_t tg = 0;
    auto at_column = [&](int j) {
        tg = (uint64_t)(epoch + (unsigned)j + 1u) << 32;
        heads = sync + SYNC_SLOTS + (int64_t)(j & 1) * PAR_WORDS;
        rows = heads + HEAD_WORDS;
    };
    auto put_head = [&]() {
        if (wv == 0 && lane < 3) {
            const uint64_t vb = (uint64_t)__double_as_longlong(gv);
            st_agent(heads + lane * LU_MAX_WG + g,
                     tg | (lane == 0 ? (vb >> 32) : (lane == 1 ? (vb & 0xffffffffu) : (uint64_t)(unsigned)gp)));
        }
    };
    // the candidate's wave: the row, and the reciprocal of its first entry
    auto send_row = [&](auto width) {
        constexpr int WD = decltype(width)::value;
        if (wv != gw) return;
        T *row = s_row[0][wv];
        if (lane == wl) put_row(row, width);
        __builtin_amdgcn_wave_barrier();
        uint64_t *mine = rows + (int64_t)g * ROW_WORDS;
        const T rc = T(1) / row[1];
        const T x = row[(lane < WD ? lane : 0) + 1];
        if constexpr (sizeof(T) == 8) {
            const uint64_t xb = (uint64_t)__double_as_longlong((double)x), rb = (uint64_t)__double_as_longlong((double)rc);
            if (lane < WD) {
                st_agent(mine + 2 * lane, tg | (xb >> 32));
                st_agent(mine + 2 * lane + 1, tg | (xb & 0xffffffffu));
            }
            if (lane < 2) st_agent(mine + 2 * 64 + lane, tg | (lane == 0 ? (rb >> 32) : (rb & 0xffffffffu)));
        } else {
            if (lane < WD) st_agent(mine + lane, tg | __float_as_uint((float)x));
            if (lane == 0) st_agent(mine + 64, tg | __float_as_uint((float)rc));
        }
    };
    auto tagged = [&](uint64_t w) { return (w >> 32) == (tg >> 32); };
    auto column = [&](int j, auto width) -> bool {
        constexpr int WD = decltype(width)::value;
        const int par = j & 1;
        if (wv == 0) {
            // the groups' candidates: lane l reads groups l and l + 64
            double cv = -2.0;
            int cp = 0x7fffffff, cg = lane;
            bool fail = false;
            int64_t spins = 0;
#pragma unroll
            for (int h = 0; h < LU_MAX_WG / 64; ++h) {
                if (h * 64 >= G) break;
                const int q = h * 64 + lane;
                const uint64_t *sl = heads + (q < G ? q : g);
                uint64_t w0, w1, w2;
                for (;;) {
                    w0 = ld_agent(sl);
                    w1 = ld_agent(sl + LU_MAX_WG);
                    w2 = ld_agent(sl + 2 * LU_MAX_WG);
                    if (__all(tagged(w0) && tagged(w1) && tagged(w2))) break;
                    if (++spins > spin_limit) {
                        fail = true;
                        break;
                    }
                }
                if (fail) break;
                const double v = __longlong_as_double((long long)((w0 << 32) | (w1 & 0xffffffffu)));
                const int x = (int)(unsigned)w2;
                if (q < G && (v > cv || (v == cv && x < cp))) {
                    cv = v;
                    cp = x;
                    cg = q;
                }
            }
            int win = 0, p = 0;
            T x = T(0), rc = T(0);
            if (!fail) {
                double best;
                const int l = wave_best(cv, cp, best, p);
                win = __builtin_amdgcn_readlane(cg, l);
                const uint64_t *row = rows + (int64_t)win * ROW_WORDS;
                const int e = lane < WD ? lane : 0;
                for (;;) {
                    bool here;
                    if constexpr (sizeof(T) == 8) {
                        const uint64_t h = ld_agent(row + 2 * e), o = ld_agent(row + 2 * e + 1);
                        const uint64_t rh = ld_agent(row + 128), ro = ld_agent(row + 129);
                        here = tagged(h) && tagged(o) && tagged(rh) && tagged(ro);
                        x = (T)__longlong_as_double((long long)((h << 32) | (o & 0xffffffffu)));
                        rc = (T)__longlong_as_double((long long)((rh << 32) | (ro & 0xffffffffu)));
                    } else {
                        const uint64_t h = ld_agent(row + e), rh = ld_agent(row + 64);
                        here = tagged(h) && tagged(rh);
                        x = (T)__uint_as_float((unsigned)h);
                        rc = (T)__uint_as_float((unsigned)rh);
                    }
                    if (__all(here)) break;
                    if (++spins > spin_limit) {
                        fail = true;
                        break;
                    }
                }
            }
            if (lane < WD) s_u[par][lane + 1] = x;
            if (lane == 0) {
                s_u[par][0] = rc;
                s_p[par] = p;
                s_own[par] = win == g ? 1 : 0;
                if (fail) s_fail = 1;
            }
        }
        __syncthreads();
        if (s_fail) return false;
        const bool more = j + 1 < kmax;
        eliminate(j, s_p[par], s_own[par] != 0, gs, s_u[par], true, width, [&](const T *x) {
            if (!more) return;
            at_column(j + 1);
            candidate(j + 1, x, [] {});
            put_head();
        });
        if (more) send_row(width);
        return true;
    };
    bool good = true;
    auto run = [&](int j, auto width) {
        if constexpr (ONE) column_one(j, width);
        else good = column(j, width);
    };
    if constexpr (!ONE) {
        T x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = a[r][0];
        at_column(0);
        candidate(0, x, [] {});
        put_head();
        send_row(std::integral_constant<int, NB>{});
    }
    int j = 0;
    if constexpr (NB == 64) {
        for (; good && j < kmax && j < 16; ++j) run(j, std::integral_constant<int, 64>{});
        for (; good && j < kmax && j < 32; ++j) run(j, std::integral_constant<int, 48>{});
    }
    if constexpr (NB >= 32)
        for (; good && j < kmax && j < NB - 16; ++j) run(j, std::integral_constant<int, 32>{});
    for (; good && j < kmax; ++j) run(j, std::integral_constant<int, NB < 16 ? NB : 16>{});
    __syncthreads();
    // a row's entries are in its own thread's column of LDS (rows of U were
    // written there by another wave, before the barrier)
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = first + t + r * NT;
        if (i < m && good) {
            const int q = pos[r] >= 0 ? pos[r] : -1 - pos[r];
            T *row = A + q;
            // live rows hold their columns of L and nothing past kmax; when
            // kmax < n every row is a row of U
            for (int c = 0; c < n; ++c) row[(int64_t)c * lda] = s_l[c][t + r * NT];
        }
    }
    if constexpr (ONE) return;
    __syncthreads();
    if (t == 0) {
        if (s_fail) st_agent(sync + SYNC_FLAG, 1);
        // the last group out moves the tags on for the next launch (every
        // group has read the epoch by then); near the end of the 32-bit range
        // the recovery launch, alone on the stream, starts them over
        const uint64_t prev = __hip_atomic_fetch_add(sync + SYNC_LEAVE, (uint64_t)1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (prev == (uint64_t)G - 1) {
            st_agent(sync + SYNC_LEAVE, 0);
            st_agent(sync + SYNC_EPOCH, (uint64_t)(epoch + (unsigned)NB));
        }
    }
}

// After every panel of several groups: nothing unless one of its waits ran
// out; then the block saved before the panel is put back, info restored, and
// the block factored by the one-work-group global-memory leaf (pivots
// rewritten).  Tags near the end of their 32-bit range start over here, on
// cleared slots, where no panel is running.
template <typename T>
__global__ __launch_bounds__(PIV_THREADS) void lu_panel_recover_kernel(int64_t m, int n, T *__restrict__ A, int64_t lda,
                                                                       int64_t *__restrict__ ipiv,
                                                                       int64_t *__restrict__ info, int64_t r0,
                                                                       uint64_t *__restrict__ sync) {
    const uint64_t flag = ld_agent(sync + SYNC_FLAG), epoch = ld_agent(sync + SYNC_EPOCH);
    if (epoch > 0xf0000000u) {
        __syncthreads();  // every wave has read the epoch
        for (int i = threadIdx.x; i < SYNC_WORDS - SYNC_SLOTS; i += PIV_THREADS) st_agent(sync + SYNC_SLOTS + i, 0);
        if (threadIdx.x == 0) st_agent(sync + SYNC_EPOCH, 0);
    }
    if (flag == 0) return;
    const T *save = reinterpret_cast<const T *>(sync + SYNC_WORDS);
    for (int64_t idx = threadIdx.x; idx < m * n; idx += PIV_THREADS) {
        const int64_t i = idx % m, c = idx / m;
        A[i + c * lda] = save[i + c * m];
    }
    if (threadIdx.x == 0) *info = (int64_t)sync[SYNC_INFO];
    __syncthreads();
    lu_leaf_body<T>(m, n, A, lda, ipiv, info, r0);
    __syncthreads();
    if (threadIdx.x == 0) st_agent(sync + SYNC_FLAG, 0);
}

__global__ void sync_zero_kernel(uint64_t *p, int words) {
    for (int i = threadIdx.x; i < words; i += blockDim.x) p[i] = 0;
}

// laswp (src/lu.jl:470): for k = k1..k2 (1-based) swap rows k and
// ipiv[k] - r0 of each of the ncols columns (ipiv holds global rows, the
// block's row 1 is global row r0 + 1); one thread per column walks the
// interchanges in order.
template <typename T>
__global__ void laswp_kernel(int64_t ncols, T *__restrict__ A, int64_t lda, int64_t k1, int64_t k2,
                             const int64_t *__restrict__ ipiv, int64_t r0) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncols) return;
    T *col = A + c * lda;
    for (int64_t k = k1; k <= k2; ++k) {
        const int64_t p = ipiv[k - 1] - 1 - r0;
        if (p != k - 1) {
            const T a = col[k - 1];
            col[k - 1] = col[p];
            col[p] = a;
        }
    }
}

// The same interchanges as one row permutation, for blocks whose rows fit
// the work-group's LDS.  Positions are taken relative to b = k1 - 1; swap k
// (0-based) exchanges positions k and p_k >= k.  Every work-group finds where
// each final row comes from and then permutes its columns.
//
// What was at position q before swap k came there with the latest earlier
// swap j that targets q (from position j before swap j, and so on from there),
// or was there from the start.  The swaps that target j all come before swap j,
// so past the first step the latest of them all is the one: head.  The first
// step needs the latest one before k with the same target: the swaps go in in
// batches of one per thread, linked by target, and each looks for its
// predecessor in its batch, or takes what head held before the batch.  Every
// position's source is then a short walk of its own, all positions at once:
// composing the swaps in order, one LDS round trip each, took 0.1 us per swap
// (430 us for the 4096 of a half of n = 8192), and without batches a matrix whose
// pivots are all the same row (a cyclic shift) cost each swap a walk along all
// of them.  Then every thread moves up to LASWP_R entries at a time, several
// columns per pass where few rows move: all loads, a barrier, the stores.
constexpr int LASWP_THREADS = 1024, LASWP_R = 16, LASWP_COLS = 4;
constexpr int LASWP_LDS = 163840 - 64;  // bytes: 4 per row of the block, 10 per swap
constexpr int LASWP_SPAN = 38912;       // rows (a source is 16 bits, and LDS holds 812 swaps beside them)
// swaps of one launch over span rows
inline int64_t laswp_swaps(int64_t span) {
    const int64_t k = (LASWP_LDS - 4 * span) / 10 / 2 * 2, most = LASWP_R * LASWP_THREADS / 2;
    return k < most ? k : most;
}

template <typename T>
__global__ __launch_bounds__(LASWP_THREADS) void laswp_perm_kernel(int64_t ncols, T *__restrict__ A, int64_t lda,
                                                                   int64_t b, int K, int span,
                                                                   const int64_t *__restrict__ ipiv, int64_t r0) {
    __shared__ __attribute__((aligned(4))) char s_mem[LASWP_LDS];
    __shared__ int s_moved;
    int *head = reinterpret_cast<int *>(s_mem);                      // position -> the last swap that targets it, -1 none
    uint16_t *piv = reinterpret_cast<uint16_t *>(s_mem + 4 * span);  // swap -> its target
    uint16_t *next = piv + K;                                        // swap -> the latest before it with the same target
    uint16_t *src = next + K;                                        // position < K -> the row that ends there
    uint16_t *dst = src + K, *dsrc = dst + K;                        // rows past K that move, and their sources
    const int t = threadIdx.x;
    constexpr uint16_t NONE = 0xffff;
    for (int x = t; x < span; x += LASWP_THREADS) head[x] = -1;
    if (t == 0) s_moved = 0;
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += LASWP_THREADS) {
        const int k = k0 + t;
        int p = k;
        if (k < K) {
            const int64_t q = ipiv[b + k] - 1 - r0 - b;
            if (q >= k && q < span) p = (int)q;  // pivots lie in [k, span)
            piv[k] = (uint16_t)p;
            if (p != k) {  // a swap with itself moves nothing
                const int old = atomicExch(&head[p], k);
                next[k] = old < 0 ? NONE : (uint16_t)old;
            }
        }
        __syncthreads();
        int before = -1;
        bool last = p != k;
        if (last) {
            for (int c = head[p]; c >= 0;) {
                if (c < k && c > before) before = c;
                if (c > k) last = false;
                if (c < k0) break;  // what the position held before this batch
                const uint16_t n = next[c];
                c = n == NONE ? -1 : (int)n;
            }
        }
        __syncthreads();  // every link of the batch has been read
        if (k < K) next[k] = before < 0 ? NONE : (uint16_t)before;
        if (last) head[p] = k;
        __syncthreads();
    }
    // the row at position q after the swaps so far that target it
    auto source = [&](int q) {
        for (int j = head[q]; j >= 0; j = head[q]) q = j;
        return q;
    };
    for (int x = t; x < span; x += LASWP_THREADS) {
        if (x < K) {
            const uint16_t j = next[x];
            src[x] = (uint16_t)(piv[x] == x ? source(x) : (j == NONE ? (int)piv[x] : source((int)j)));
        } else if (head[x] >= 0) {
            const int from = source(x);
            if (from != x) {
                const int at = atomicAdd(&s_moved, 1);
                dst[at] = (uint16_t)x;
                dsrc[at] = (uint16_t)from;
            }
        }
    }
    __syncthreads();
    const int tot = K + s_moved;
    auto to = [&](int i) { return i < K ? i : (int)dst[i - K]; };
    auto from = [&](int i) { return i < K ? (int)src[i] : (int)dsrc[i - K]; };
    if (tot <= LASWP_THREADS) {
        const int w = (tot + 63) / 64 * 64, cpp = LASWP_THREADS / w;  // threads per column, columns side by side
        const int i = t % w, side = t / w;
        const bool on = side < cpp && i < tot;
        const int x = on ? to(i) : 0, y = on ? from(i) : 0;
        const bool move = on && x != y;
        for (int64_t c0 = (int64_t)blockIdx.x * cpp * LASWP_COLS; c0 < ncols; c0 += (int64_t)gridDim.x * cpp * LASWP_COLS) {
            T v[LASWP_COLS];
#pragma unroll
            for (int u = 0; u < LASWP_COLS; ++u) {
                const int64_t c = c0 + u * cpp + side;
                v[u] = move && c < ncols ? A[c * lda + b + y] : T(0);
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < LASWP_COLS; ++u) {
                const int64_t c = c0 + u * cpp + side;
                if (move && c < ncols) A[c * lda + b + x] = v[u];
            }
        }
        return;
    }
    for (int64_t c = blockIdx.x; c < ncols; c += gridDim.x) {
        T *col = A + c * lda + b;
        T v[LASWP_R];
#pragma unroll
        for (int r = 0; r < LASWP_R; ++r) {
            const int i = t + r * LASWP_THREADS;
            v[r] = (i < tot) ? col[from(i)] : T(0);
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < LASWP_R; ++r) {
            const int i = t + r * LASWP_THREADS;
            if (i < tot && from(i) != to(i)) col[to(i)] = v[r];
        }
    }
}

// A12 = L11^-1 A12 for a unit lower L11 of n1 <= SMALL_TRSM rows (the
// reference's trsm!('L','L','N','U'), src/lu.jl:277): forward substitution,
// one thread per column of A12 holding it in registers; L11 is read through
// the cache (every thread reads the same entries).  Replaces the inverse and
// panel launches of the general TRSM at the bottom of the recursion.
constexpr int SMALL_TRSM = 32;

template <typename T>
__global__ __launch_bounds__(64) void lu_trsm_small_kernel(int n1, int64_t n2, const T *__restrict__ L, int64_t lda,
                                                           T *__restrict__ B) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n2) return;
    T *b = B + c * lda;
    T x[SMALL_TRSM];
#pragma unroll
    for (int i = 0; i < SMALL_TRSM; ++i) x[i] = b[i < n1 ? i : 0];
#pragma unroll
    for (int k = 0; k < SMALL_TRSM - 1; ++k) {
        const T xk = x[k];
        const T *lk = L + (int64_t)(k < n1 ? k : 0) * lda;
#pragma unroll
        for (int i = k + 1; i < SMALL_TRSM; ++i)
            if (i < n1) x[i] -= lk[i] * xk;
    }
#pragma unroll
    for (int i = 0; i < SMALL_TRSM; ++i)
        if (i < n1) b[i] = x[i];
}

__global__ void info_zero_kernel(int64_t *info) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *info = 0;
}

// Exchange slots and saved block of the register panels, two buffers per
// (device, stream), one for panels of up to SMALL_ROWS rows (2.4 MB) and one for
// taller ones (8.7 MB), each allocated when first needed and kept: launches on
// one stream run in order, so they share it.  A panel and the recovery launch
// that follows it are enqueued under the lock: with another host thread's panel
// in between, the recovery would find that panel's block saved.
constexpr int64_t SMALL_ROWS = 4096;
struct PanelSync {
    int dev;
    hipStream_t stream;
    std::thread::id thread;  // hipStreamPerThread is another stream in every thread
    uint64_t *ptr[2] = {nullptr, nullptr};
    std::mutex mu;
};

PanelSync *panel_sync(hipStream_t s, int32_t *st) {
    static std::mutex mu;
    static std::vector<std::unique_ptr<PanelSync>> cache;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *st = report_hip(e, "lu panel device");
        return nullptr;
    }
    const std::thread::id me = s == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id();
    std::lock_guard<std::mutex> g(mu);
    for (auto &c : cache)
        if (c->dev == dev && c->stream == s && c->thread == me) return c.get();
    cache.emplace_back(new PanelSync());
    cache.back()->dev = dev;
    cache.back()->stream = s;
    cache.back()->thread = me;
    return cache.back().get();
}

// The buffer for m rows, called with sync->mu held.
uint64_t *panel_buffer(PanelSync *sync, int64_t m, int32_t *st) {
    uint64_t *&p = sync->ptr[m <= SMALL_ROWS ? 0 : 1];
    if (p != nullptr) return p;
    uint64_t *q = nullptr;
    const int64_t save = m <= SMALL_ROWS ? SMALL_ROWS * 64 * 8 : SAVE_BYTES;
    hipError_t e = hipMalloc((void **)&q, SYNC_WORDS * 8 + save);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(sync_zero_kernel, dim3(1), dim3(256), 0, sync->stream, q, SYNC_WORDS);
        e = hipGetLastError();
    }
    if (e != hipSuccess) {
        *st = report_hip(e, "lu panel sync buffer");
        return nullptr;
    }
    return p = q;
}

bool is_captured(hipStream_t s) {
    if (s == nullptr) return false;  // the null stream cannot be
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return st != hipStreamCaptureStatusNone;
}

template <typename T>
struct LuRec {
    int32_t dtype;
    int64_t lda;
    int64_t *info;
    hipStream_t s;
    int32_t st = NLA_OK;
    int64_t split_rows = lu_split_rows();
    bool stateless = false;  // blocks of 129 to REG_ROWS rows in the register leaf: nothing shared, nothing allocated
    int64_t spin_limit = lu_spin_limit() > 0 ? lu_spin_limit() : SPLIT_SPIN_LIMIT;

    // the register panel for up to MOST rows
    template <int NB, int R, int NT, int MOST>
    void panel_of(int64_t m, int n, T *A, int64_t *ipiv, int64_t r0) {
        constexpr int GROUPS = MOST / (NT * R), PER_CU = 163840 / (NB * NT * R * (int)sizeof(T) + 6144);
        static_assert(GROUPS <= LU_MAX_WG && GROUPS <= LU_CUS * PER_CU, "every group gets a place");
        const unsigned g = (unsigned)((m + NT * R - 1) / (NT * R));
        if (g == 1) {
            hipLaunchKernelGGL((lu_panel_kernel<T, NB, R, NT, true>), dim3(1), dim3(NT), 0, s, (int)m, n, A, lda, ipiv,
                               info, r0, (uint64_t *)nullptr, (int64_t)0);
            ok(hipGetLastError(), "lu panel");
            return;
        }
        PanelSync *sync = panel_sync(s, &st);
        if (!sync) return;
        std::lock_guard<std::mutex> pair(sync->mu);
        uint64_t *buf = panel_buffer(sync, m, &st);
        if (!buf) return;
        hipLaunchKernelGGL((lu_panel_kernel<T, NB, R, NT, false>), dim3(g), dim3(NT), 0, s, (int)m, n, A, lda, ipiv,
                           info, r0, buf, spin_limit);
        if (!ok(hipGetLastError(), "lu panel")) return;
        hipLaunchKernelGGL(lu_panel_recover_kernel<T>, dim3(1), dim3(PIV_THREADS), 0, s, m, n, A, lda, ipiv, info, r0,
                           buf);
        ok(hipGetLastError(), "lu panel recovery");
    }

    // Few columns of more rows than a single group's panel takes (128): one
    // group of the register leaf against a panel of several and its recovery
    // launch.  Measured on MI355X (us per call, leaf / panel): FP64 256 x 1
    // 6.2 / 10.3, 256 x 8 25.8 / 30.3, 1000 x 8 29.2 / 30.1, 2048 x 4
    // 18.4 / 19.2, 2048 x 8 33.2 / 29.5, 4096 x 1 7.0 / 10.7, 4096 x 4
    // 21.8 / 19.8; FP32 1000 x 8 25.7 / 27.9, 2048 x 8 28.9 / 26.9.
    static bool narrow(int64_t m, int64_t n) {
        return n <= LEAF_COLS && m > 128 && m <= REG_ROWS && m * n <= 12288;
    }

    // an m x n panel, n <= panel_cols(m): 128-row groups up to 8192 rows (each
    // lane polls one group), 256 rows and more above
    void panel(int64_t m, int n, T *A, int64_t *ipiv, int64_t r0) {
        const int nb = panel_cols<T>(m);
        if constexpr (sizeof(T) == 8) {
            if (nb == 64 && m <= 8192) panel_of<64, 1, 128, 8192>(m, n, A, ipiv, r0);
            else if (nb == 64) panel_of<64, 1, 256, 16384>(m, n, A, ipiv, r0);
            else if (nb == 32) panel_of<32, 1, 256, 32768>(m, n, A, ipiv, r0);
            else if (nb == 16) panel_of<16, 2, 256, 65536>(m, n, A, ipiv, r0);
            else panel_of<8, 4, 256, 131072>(m, n, A, ipiv, r0);
        } else {
            if (nb == 64 && m <= 8192) panel_of<64, 1, 128, 8192>(m, n, A, ipiv, r0);
            else if (nb == 64) panel_of<64, 1, 256, 32768>(m, n, A, ipiv, r0);
            else if (nb == 32) panel_of<32, 2, 256, 65536>(m, n, A, ipiv, r0);
            else panel_of<16, 4, 256, 131072>(m, n, A, ipiv, r0);
        }
    }

    bool ok(hipError_t e, const char *where) {
        if (e != hipSuccess && st == NLA_OK) st = report_hip(e, where);
        return st == NLA_OK;
    }

    // interchanges k1..k2 of the m-row block at A on ncols columns: as
    // permutations of what fits LDS, else the sequential walk
    void laswp(T *A, int64_t m, int64_t ncols, int64_t k1, int64_t k2, const int64_t *ipiv, int64_t r0) {
        if (ncols <= 0) return;
        while (k1 <= k2 && st == NLA_OK) {
            const int64_t b = k1 - 1, span = m - b;
            if (span > LASWP_SPAN) {
                hipLaunchKernelGGL(laswp_kernel<T>, dim3((unsigned)((ncols + 63) / 64)), dim3(64), 0, s, ncols, A, lda,
                                   k1, k2, ipiv, r0);
                ok(hipGetLastError(), "laswp");
                return;
            }
            const int64_t K = std::min(k2 - b, laswp_swaps(span));
            const int64_t per = K <= LASWP_THREADS / 2 ? LASWP_THREADS / (2 * K) * LASWP_COLS : 1;  // columns of a pass
            const unsigned g = (unsigned)std::min<int64_t>((ncols + per - 1) / per, 512);
            hipLaunchKernelGGL(laswp_perm_kernel<T>, dim3(g), dim3(LASWP_THREADS), 0, s, ncols, A, lda, b, (int)K,
                               (int)span, ipiv, r0);
            ok(hipGetLastError(), "laswp");
            k1 += K;
        }
    }

    // The whole factorization.  A captured call must not allocate, and its
    // graph may run beside others of its stream: its blocks of up to REG_ROWS
    // rows take no exchange buffer if the stream has none for them yet, or if
    // the call is thin (up to 65 columns; past them it has a triangular solve,
    // whose workspace is the stream's in any case).  The register leaf takes up
    // to 3 times as long as the panels there (1000 x 64 FP64 420 / 166 us).
    void run(int64_t m, int64_t n, T *A, int64_t *ipiv) {
        if (is_captured(s)) {
            PanelSync *sync = panel_sync(s, &st);
            if (!sync) return;
            std::lock_guard<std::mutex> g(sync->mu);
            stateless = (m <= REG_ROWS && std::min(m, n) <= 65) || sync->ptr[0] == nullptr;
        }
        rec(m, n, A, ipiv, 0);
    }

    // Factor the m x n block at A, whose first row and column are the global
    // row / column r0 (blocks start on the diagonal); its pivots go to
    // ipiv[0 .. min(m,n)) as global 1-based rows, which is what the
    // reference's "ipiv[i] += n1" (src/lu.jl:289-291) makes of them.
    void rec(int64_t m, int64_t n, T *A, int64_t *ipiv, int64_t r0) {
        if (st != NLA_OK || m == 0 || n == 0) return;
        const bool regs = split_rows > 0 && m >= split_rows, leaf = m > 128 && m <= REG_ROWS && stateless;
        const int nb = regs && !leaf ? panel_cols<T>(m) : 0;
        if (regs && (leaf ? n <= LEAF_COLS : narrow(m, n))) {
            hipLaunchKernelGGL(lu_leaf_reg_kernel<T>, dim3(1), dim3(REG_THREADS), 0, s, (int)m, (int)n, A, lda, ipiv,
                               info, r0);
            ok(hipGetLastError(), "lu register leaf");
            return;
        }
        if (n <= nb) {
            panel(m, (int)n, A, ipiv, r0);
            return;
        }
        if (n <= LEAF_COLS || m == 1) {
            const int nl = (int)(n <= LEAF_COLS ? n : 1);  // m == 1: only the first column is examined
            hipLaunchKernelGGL(lu_leaf_kernel<T>, dim3(1), dim3(PIV_THREADS), 0, s, m, nl, A, lda, ipiv, info, r0);
            ok(hipGetLastError(), "lu leaf");
            return;
        }
        // whole panels on the left: n1 is half of the columns rounded up to a
        // multiple of the panel's width (all of a block of at most nb rows)
        const int64_t mn = m < n ? m : n, half = nb > 0 ? ((mn + 1) / 2 + nb - 1) / nb * nb : mn / 2;
        const int64_t n1 = half < mn ? half : (mn < n ? mn : mn / 2), n2 = n - n1;
        rec(m, n1, A, ipiv, r0);
        laswp(A + n1 * lda, m, n2, 1, n1, ipiv, r0);
        if (st != NLA_OK) return;
        // A12 = L11^-1 A12 (unit lower; the identity for one column)
        if (n1 > 1 && n1 <= SMALL_TRSM) {
            hipLaunchKernelGGL(lu_trsm_small_kernel<T>, dim3((unsigned)((n2 + 63) / 64)), dim3(64), 0, s, (int)n1, n2,
                               A, lda, A + n1 * lda);
            if (!ok(hipGetLastError(), "lu small trsm")) return;
        } else if (n1 > 1) {
            const int32_t r = nla_trsm('L', 'L', 'N', 'U', dtype, 1.0, n1, n2, A, lda, A + n1 * lda, lda, s);
            if (r != NLA_OK) {
                st = r;
                return;
            }
        }
        // A22 -= A21 A12
        if (m <= n1) return;
        {
            const int32_t r = nla_gemm(dtype, 'N', 'N', m - n1, n2, n1, -1.0, A + n1, lda, A + n1 * lda, lda, 1.0,
                                       A + n1 + n1 * lda, lda, s);
            if (r != NLA_OK) {
                st = r;
                return;
            }
        }
        rec(m - n1, n2, A + n1 + n1 * lda, ipiv + n1, r0 + n1);
        laswp(A, m, n1, n1 + 1, mn, ipiv, r0);
    }
};

}  // namespace
}  // namespace nla

using namespace nla;

extern "C" int32_t nla_getrf2(int32_t dtype, int64_t m, int64_t n, void *A, int64_t lda, int64_t *ipiv,
                              int64_t *info, void *stream) {
    if (dtype != NLA_F32 && dtype != NLA_F64) return report_bad_arg(1, "dtype");
    if (m < 0) return report_bad_arg(2, "m");
    if (n < 0) return report_bad_arg(3, "n");
    if (lda < (m > 1 ? m : 1)) return report_bad_arg(5, "lda");
    if (m > 0 && n > 0 && A == nullptr) return report_bad_arg(4, "A");
    if (m > 0 && n > 0 && ipiv == nullptr) return report_bad_arg(6, "ipiv");
    if (info == nullptr) return report_bad_arg(7, "info");
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(info_zero_kernel, dim3(1), dim3(64), 0, s, info);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return report_hip(e, "getrf2 info");
    if (m == 0 || n == 0) return NLA_OK;
    if (dtype == NLA_F64) {
        LuRec<double> r{dtype, lda, info, s};
        r.run(m, n, (double *)A, ipiv);
        return r.st;
    }
    LuRec<float> r{dtype, lda, info, s};
    r.run(m, n, (float *)A, ipiv);
    return r.st;
}
