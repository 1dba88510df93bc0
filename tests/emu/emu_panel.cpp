// The dispatch of the panels (launch_panel of nla_panel.hip) on the CPU: which
// kernel a panel takes and with how many groups, without running it.
#include <cstdio>
#include <string>

#define hipLaunchKernelGGL(kernel, grid, block, ...) emu_launch(#kernel, grid, block)
#include "hip/hip_runtime.h"
static std::string g_log;
static void emu_launch(const char *name, dim3 grid, dim3 block) {
    g_log = std::to_string(grid.x) + " " + std::to_string(block.x) + " " + name;
}
inline hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
// kernels that are named by address are compiled here too, but never run
#include <cstdlib>
#define asm
#define volatile(...)
inline unsigned atomicMax(unsigned *p, unsigned v) { return *p = *p > v ? *p : v; }
#include "../../nextla.jl_amd/csrc/nla_panel.hip"

namespace {
template <typename T>
int launch(int trmm, int n, int64_t m, int kc, int bcol, int unit, int strip, int waves) {
    static T mem[4];
    nla::PanelArgs<T> a{};
    a.trmm = trmm != 0;
    a.lower = true;
    a.nbig = n;
    a.m = m;
    a.M = mem;
    a.mrs = kc ? 4096 : 1;
    a.mcs = kc ? 1 : 4096;
    a.B = mem;
    a.brs = bcol ? 1 << 20 : 1;
    a.bcs = bcol ? 1 : 4096;
    a.scale = T(1);
    a.unit = unit != 0;
    a.strip = strip;
    a.waves = waves;
    g_log.clear();
    return (int)nla::launch_panel<T>(a, nullptr);
}
}  // namespace

// "groups threads kernel" of the panel's launch.
extern "C" int emu_panel(int dtype, int trmm, int n, int64_t m, int kc, int bcol, int unit, int strip, int waves,
                         char *out, int64_t cap) {
    const int r = dtype == 1 ? launch<double>(trmm, n, m, kc, bcol, unit, strip, waves)
                             : launch<float>(trmm, n, m, kc, bcol, unit, strip, waves);
    snprintf(out, (size_t)cap, "%s", g_log.c_str());
    return r;
}
