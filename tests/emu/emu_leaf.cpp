// The 64-block inverse's kernel on the CPU (see hip/hip_runtime.h here).
#include "../../nextla.jl_amd/csrc/nla_leaf.hip"

namespace {
template <typename T>
int trtri64(int64_t n, const T *A, int64_t rs, int64_t cs, int lower, int unit, T *W, int *F, const int *order) {
    const std::vector<int> waves(order, order + 4);
    for (int b = 0; b < (int)((n + 63) / 64); ++b)
        if (!emu::run(256, b, (int)((n + 63) / 64), waves,
                      [&] { nla::trtri64_kernel<T>(n, A, rs, cs, lower, unit, W, F); }))
            return 1;
    return 0;
}
}  // namespace

extern "C" int emu_trtri64_f64(int64_t n, const double *A, int64_t rs, int64_t cs, int lower, int unit, double *W,
                               int *F, const int *order) {
    return trtri64<double>(n, A, rs, cs, lower, unit, W, F, order);
}
extern "C" int emu_trtri64_f32(int64_t n, const float *A, int64_t rs, int64_t cs, int lower, int unit, float *W, int *F,
                               const int *order) {
    return trtri64<float>(n, A, rs, cs, lower, unit, W, F, order);
}
