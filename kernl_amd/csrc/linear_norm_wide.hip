// linear + residual + LayerNorm in one launch on the 256-row wide kernel (norm_exchange.h says how the workgroups of a row agree).
#include "linear_wide_norm.h"

namespace kernl {

template <typename T, int NBN>
static void launch_wide_norm(const LinearArgs &a, const NormExchange &norm) {
    auto kern = linear_wide_kernel<T, KERNL_ACT_NONE, NBN, false, false, false, false, NormExchange>;
    static bool attr_done = false;  // benign race: the attribute call is idempotent
    if (!attr_done) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kWideNormLds);
        attr_done = true;
    }
    const int tiles_m = (a.M + 255) / 256, tiles_n = a.N / (32 * NBN);
    const T *bias = static_cast<const T *>(a.bias);
    hipLaunchKernelGGL(kern, dim3((tiles_m * tiles_n + 7) / 8 * 8), dim3(256), kWideNormLds, a.st, static_cast<const T *>(a.x),
                       static_cast<const T *>(a.w), bias, static_cast<T *>(a.out), (T *)nullptr, a.M, a.N, a.K, a.x_rs, a.out_rs, (int64_t)1,
                       (int64_t)0, (int64_t)0, tiles_m, tiles_n, 1, 0, bias != nullptr && aligned16(bias), (const float *)nullptr, norm);
}

void run_wide_norm(const LinearArgs &a, int dtype, int cols, const NormExchange &norm) {
    if (dtype == KERNL_F16) cols == 192 ? launch_wide_norm<f16, 6>(a, norm) : launch_wide_norm<f16, 8>(a, norm);
    else cols == 192 ? launch_wide_norm<bf16, 6>(a, norm) : launch_wide_norm<bf16, 8>(a, norm);
}

}  // namespace kernl
