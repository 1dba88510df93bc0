// The host side of nla_getrf2 on the CPU: the launches that it makes, in the
// order in which they reach a stream, without running them.
#include <chrono>
#include <cstdio>
#include <mutex>
#include <string>
#include <thread>

#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...) emu_launch(#kernel, grid, stream)
namespace {
struct Log {
    std::mutex mu;
    std::string text;
    int next_thread = 0;
    int capturing = 0, mallocs = 0;
    int64_t bytes = 0;
} g_log;
int thread_number() {
    static thread_local int me = [] {
        std::lock_guard<std::mutex> g(g_log.mu);
        return g_log.next_thread++;
    }();
    return me;
}
}  // namespace

#include "hip/hip_runtime.h"

// a launch takes a moment, so that another thread's may come in between
template <typename... Ts>
static void emu_launch(const char *name, dim3 grid, Ts...) {
    const int me = thread_number();
    {
        std::lock_guard<std::mutex> g(g_log.mu);
        g_log.text += std::to_string(me) + " " + std::to_string(grid.x) + " " + name + "\n";
    }
    std::this_thread::sleep_for(std::chrono::microseconds(300));
}
hipError_t hipGetDevice(int *dev) {
    *dev = 0;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    if (g_log.capturing) return hipErrorStreamCaptureUnsupported;
    ++g_log.mallocs;
    g_log.bytes += (int64_t)bytes;
    *p = (void *)(uintptr_t)(4096 * (size_t)g_log.mallocs);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) {
    *st = g_log.capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}

#include "../../nextla.jl_amd/csrc/nla_lu.hip"

namespace nla {
int32_t report_hip(hipError_t e, const char *) { return e == hipSuccess ? 0 : -1000; }
int32_t report_bad_arg(int k, const char *) { return -k; }
int lu_split_rows() { return 1; }
int lu_spin_limit() { return 0; }
}  // namespace nla
extern "C" {
int32_t nla_trsm(char, char, char, char, int32_t, double, int64_t, int64_t, const void *, int64_t, void *, int64_t,
                 void *) {
    emu_launch("nla_trsm", dim3(1));
    return 0;
}
int32_t nla_gemm(int32_t, char, char, int64_t, int64_t, int64_t, double, const void *, int64_t, const void *, int64_t,
                 double, void *, int64_t, void *) {
    emu_launch("nla_gemm", dim3(1));
    return 0;
}

// One LU of m x n by each of `threads` host threads on the same stream; the
// launches as lines "thread groups kernel".
int emu_getrf2(int dtype, int64_t m, int64_t n, int threads, int64_t stream, int capturing, char *out, int64_t cap) {
    g_log.text.clear();
    g_log.capturing = capturing;
    g_log.next_thread = 0;
    int64_t ipiv = 0, info = 0;
    double A = 0;
    std::vector<std::thread> pool;
    std::vector<int> st((size_t)threads, 0);
    for (int i = 0; i < threads; ++i)
        pool.emplace_back([&, i] {
            st[(size_t)i] = nla_getrf2(dtype, m, n, &A, m, &ipiv, &info, (void *)stream);
        });
    for (auto &t : pool) t.join();
    g_log.capturing = 0;
    snprintf(out, (size_t)cap, "%s", g_log.text.c_str());
    for (int s : st)
        if (s != 0) return s;
    return 0;
}
// Interchanges b + 1 .. b + K (1-based rows in ipiv) of one block of rows on
// the device kernel, its waves in either order.
int emu_laswp(int64_t ncols, double *A, int64_t lda, int64_t b, int K, int span, const int64_t *ipiv, int reversed) {
    std::vector<int> order;
    for (int w = 0; w < nla::LASWP_THREADS / 64; ++w) order.push_back(reversed ? nla::LASWP_THREADS / 64 - 1 - w : w);
    return emu::run(nla::LASWP_THREADS, 0, 1, order,
                    [&] { nla::laswp_perm_kernel<double>(ncols, A, lda, b, K, span, ipiv, 0); })
               ? 0
               : 1;
}
int64_t emu_allocated(void) { return g_log.bytes; }
}
