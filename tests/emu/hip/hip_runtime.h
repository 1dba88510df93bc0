// A stand-in for HIP's runtime header that runs a kernel's source on the CPU,
// for tests of what depends on the order of its waves: every thread of one
// work-group is a fiber, a wave runs until all of its lanes wait, and the
// waves take turns in an order that the caller gives, so that the first of
// them is always as far ahead of the others as the barriers let it be.
// Wave-wide operations (shuffles, votes, MFMA, wave barriers) are points where
// a wave's 64 lanes meet; whole waves must reach them.  One work-group at a
// time: shared arrays are static.
#pragma once

#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <cmath>
#include <functional>
#include <limits>
#include <memory>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(...)
#define __align__(n) __attribute__((aligned(n)))
#ifndef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) ((void)0)
#endif

typedef void *hipStream_t;
#define hipStreamPerThread ((hipStream_t)2)
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorStreamCaptureUnsupported = 900 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };
inline hipError_t hipGetLastError() { return hipSuccess; }
// for host code under test: what it allocates, and whether the stream is captured
hipError_t hipGetDevice(int *dev);
hipError_t hipMalloc(void **p, size_t bytes);
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st);
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct int2 {
    int x, y;
};
using std::fabs;
using std::fma;

namespace emu {

struct Wave {
    unsigned char buf[2][64][64];
    int arrived = 0;
    unsigned gen = 0;
};
struct Fiber {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    const unsigned *wait = nullptr;  // runnable when *wait has left waitgen
    unsigned waitgen = 0;
    bool done = false;
};
struct Group {
    int nt = 0, block = 0, grid = 1, cur = 0, live = 0, arrived = 0;
    unsigned gen = 0;
    std::vector<Fiber> fibers;
    std::vector<Wave> waves;
    ucontext_t main;
    std::function<void()> kernel;
};
inline Group *&group() {
    static Group *g = nullptr;
    return g;
}
inline void wait_on(const unsigned *gen) {
    Group &g = *group();
    Fiber &f = g.fibers[(size_t)g.cur];
    f.wait = gen;
    f.waitgen = *gen;
    swapcontext(&f.ctx, &g.main);
    f.wait = nullptr;
}
inline void sync_block() {
    Group &g = *group();
    if (++g.arrived == g.live) {
        g.arrived = 0;
        ++g.gen;
    } else {
        wait_on(&g.gen);
    }
}
// every lane's v, by lane
template <typename V>
struct Lanes {
    V v[64];
};
template <typename V>
inline Lanes<V> meet(V v) {
    static_assert(sizeof(V) <= 64, "a lane's value");
    Group &g = *group();
    Wave &w = g.waves[(size_t)g.cur / 64];
    const unsigned par = w.gen & 1;
    memcpy(w.buf[par][g.cur % 64], &v, sizeof(V));
    if (++w.arrived == 64) {
        w.arrived = 0;
        ++w.gen;
    } else {
        wait_on(&w.gen);
    }
    Lanes<V> all;
    for (int l = 0; l < 64; ++l) memcpy(&all.v[l], w.buf[par][l], sizeof(V));
    return all;
}
inline void entry() {
    Group &g = *group();
    const int me = g.cur;
    g.kernel();
    g.fibers[(size_t)me].done = true;
    if (--g.live > 0 && g.arrived == g.live) {  // a barrier does not wait for threads that have left
        g.arrived = 0;
        ++g.gen;
    }
    swapcontext(&g.fibers[(size_t)me].ctx, &g.main);
}
// One work-group of nt threads; order: the waves, first the one that runs
// ahead.  False if its threads wait for each other for ever.
inline bool run(int nt, int block, int grid, const std::vector<int> &order, std::function<void()> kernel) {
    Group g;
    group() = &g;
    g.nt = g.live = nt;
    g.block = block;
    g.grid = grid;
    g.kernel = std::move(kernel);
    g.fibers.resize((size_t)nt);
    g.waves.resize((size_t)(nt + 63) / 64);
    constexpr size_t STACK = 1 << 17;
    for (auto &f : g.fibers) {
        f.stack.reset(new char[STACK]);
        getcontext(&f.ctx);
        f.ctx.uc_stack.ss_sp = f.stack.get();
        f.ctx.uc_stack.ss_size = STACK;
        f.ctx.uc_link = &g.main;
        makecontext(&f.ctx, entry, 0);
    }
    for (;;) {
        bool moved = false;
        for (int w : order) {
            bool any;
            do {
                any = false;
                for (int t = 64 * w; t < 64 * w + 64 && t < nt; ++t) {
                    Fiber &f = g.fibers[(size_t)t];
                    if (f.done || (f.wait != nullptr && *f.wait == f.waitgen)) continue;
                    g.cur = t;
                    swapcontext(&g.main, &f.ctx);
                    any = moved = true;
                }
            } while (any);
        }
        if (!moved) break;
    }
    group() = nullptr;
    return g.live == 0;
}
inline dim3 tid() { return dim3((unsigned)group()->cur, 0, 0); }
inline int lane() { return group()->cur % 64; }
inline int lane_of(int v, int l) { return meet(v).v[l]; }

// D = A B + C in the lane layouts of the MFMA instructions, with fused steps in ascending k
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16 __attribute__((ext_vector_type(16)));
template <typename T, typename V>
inline V mfma_16x16x4(T a, T b, V c, int istep, int rstep) {
    const Lanes<T> A = meet(a), B = meet(b);
    const int l = lane();
    for (int r = 0; r < 4; ++r) {
        const int i = istep * (l / 16) + rstep * r, j = l % 16;
        T x = c[r];
        for (int k = 0; k < 4; ++k) x = std::fma(A.v[i + 16 * k], B.v[j + 16 * k], x);
        c[r] = x;
    }
    return c;
}
inline f16 mfma_32x32x2(float a, float b, f16 c) {
    const Lanes<float> A = meet(a), B = meet(b);
    const int l = lane();
    for (int r = 0; r < 16; ++r) {
        const int i = 8 * (r / 4) + 4 * (l / 32) + r % 4, j = l % 32;
        float x = c[r];
        for (int k = 0; k < 2; ++k) x = std::fma(A.v[i + 32 * k], B.v[j + 32 * k], x);
        c[r] = x;
    }
    return c;
}

}  // namespace emu

#define threadIdx (emu::tid())
#define blockIdx (dim3((unsigned)emu::group()->block, 0, 0))
#define gridDim (dim3((unsigned)emu::group()->grid))
#define blockDim (dim3((unsigned)emu::group()->nt))

inline void __syncthreads() { emu::sync_block(); }
template <typename T>
inline T __shfl_xor(T v, int o, int = 64) {
    return emu::meet(v).v[emu::lane() ^ o];
}
inline int __all(int p) {
    const auto v = emu::meet(p);
    for (int l = 0; l < 64; ++l)
        if (!v.v[l]) return 0;
    return 1;
}
inline unsigned long long __ballot(int p) {
    const auto v = emu::meet(p);
    unsigned long long m = 0;
    for (int l = 0; l < 64; ++l) m |= (unsigned long long)(v.v[l] != 0) << l;
    return m;
}
inline int __ffsll(unsigned long long v) { return __builtin_ffsll((long long)v); }
template <typename To, typename From>
inline To emu_bits(From v) {
    static_assert(sizeof(To) == sizeof(From), "the same bits");
    To r;
    memcpy(&r, &v, sizeof(To));
    return r;
}
inline long long __double_as_longlong(double v) { return emu_bits<long long>(v); }
inline double __longlong_as_double(long long v) { return emu_bits<double>(v); }
inline unsigned __float_as_uint(float v) { return emu_bits<unsigned>(v); }
inline float __uint_as_float(unsigned v) { return emu_bits<float>(v); }
using std::fmax;
template <typename T>
inline T atomicExch(T *p, T v) {
    const T old = *p;
    *p = v;
    return old;
}
template <typename T>
inline T atomicAdd(T *p, T v) {
    const T old = *p;
    *p = old + v;
    return old;
}

#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) (emu::mfma_16x16x4<double, emu::d4>(a, b, c, 1, 4))
#define __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, x, y, z) (emu::mfma_16x16x4<float, emu::f4>(a, b, c, 4, 1))
#define __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, x, y, z) (emu::mfma_32x32x2(a, b, c))
#define __builtin_amdgcn_wave_barrier() ((void)emu::meet(0))
#define __builtin_amdgcn_sched_barrier(m) ((void)0)
#define __builtin_amdgcn_s_setprio(p) ((void)0)
#define __builtin_amdgcn_readlane(x, l) (emu::lane_of((int)(x), l))
#define __builtin_amdgcn_readfirstlane(x) (emu::lane_of((int)(x), 0))
// lane moves of DPP; not modelled
#define __builtin_amdgcn_update_dpp(old, v, ctrl, rows, banks, bound) (abort(), (v))
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_store(p, v, order, scope) ((void)(*(p) = (v)))
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_fetch_add(p, v, order, scope) (atomicAdd((p), (v)))
