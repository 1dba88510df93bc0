// lauum's product kernels on the CPU (see hip/hip_runtime.h here).
#include "../../nextla.jl_amd/csrc/nla_lauum.hip"

namespace nla {
int32_t report_hip(hipError_t e, const char *) { return (int)e; }
int32_t report_bad_arg(int k, const char *) { return -k; }
}  // namespace nla

namespace {
template <typename T, int RB, bool LOWER>
int product(int64_t n, T *A, int64_t lda) {
    constexpr int B = 16 * RB;
    const int64_t t = (n + B - 1) / B, total = t * (t + 1) / 2;
    std::vector<T> W((size_t)(total * B * B));
    for (int b = 0; b < (int)total; ++b)
        if (!emu::run(nla::LAUUM_KS * 64, b, (int)total, {0, 1, 2, 3},
                      [&] { nla::lauum_product_kernel<T, RB, LOWER>(n, A, lda, W.data(), 0); }))
            return 1;
    for (int b = 0; b < (int)total; ++b)
        if (!emu::run(256, b, (int)total, {0, 1, 2, 3},
                      [&] { nla::lauum_store_kernel<T, B, LOWER>(n, A, lda, W.data(), 0); }))
            return 1;
    return 0;
}
template <typename T>
int lauum(int lower, int large, int64_t n, T *A, int64_t lda) {
    if (large) return lower ? product<T, 4, true>(n, A, lda) : product<T, 4, false>(n, A, lda);
    return lower ? product<T, 2, true>(n, A, lda) : product<T, 2, false>(n, A, lda);
}
}  // namespace

extern "C" int emu_lauum_f64(int lower, int large, int64_t n, double *A, int64_t lda) {
    return lauum<double>(lower, large, n, A, lda);
}
extern "C" int emu_lauum_f32(int lower, int large, int64_t n, float *A, int64_t lda) {
    return lauum<float>(lower, large, n, A, lda);
}
