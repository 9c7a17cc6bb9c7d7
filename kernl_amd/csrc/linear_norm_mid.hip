// linear + residual + LayerNorm in one launch on the tiles of linear_mid.h (norm_exchange.h says how the workgroups of a row agree).
#include "linear_mid.h"

namespace kernl {

template <typename T, typename Cfg>
__global__ void __launch_bounds__(Cfg::WAVES * 64, Cfg::WAVES / 4)
linear_mid_norm_kernel(const T *__restrict__ X, const T *__restrict__ W, const T *__restrict__ bias, T *__restrict__ out, int M, int N, int K,
                       int64_t ldx, int64_t out_rs, int tiles_m, MidGrid grid, NormExchange norm) {
    linear_mid_tile<T, Cfg, false>(X, W, bias, out, (T *)nullptr, nullptr, (const T *)nullptr, M, N, K, ldx, out_rs, 1, 0, 0, 0, 0, KERNL_ACT_NONE,
                                   tiles_m, grid, nullptr, 0, 0, norm);
}

template <typename T, typename Cfg>
static void launch_mid_norm(const LinearArgs &a, const NormExchange &norm) {
    auto kern = linear_mid_norm_kernel<T, Cfg>;
    static bool attr_done = false;  // benign race: the attribute call is idempotent
    if (!attr_done) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS);
        attr_done = true;
    }
    const int tiles_m = (a.M + Cfg::BM - 1) / Cfg::BM, tiles_n = a.N / Cfg::BN;
    MidGrid grid;
    const int blocks = mid_grid<Cfg>(tiles_m, tiles_n, 1, grid);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(Cfg::WAVES * 64), Cfg::LDS, a.st, static_cast<const T *>(a.x), static_cast<const T *>(a.w),
                       static_cast<const T *>(a.bias), static_cast<T *>(a.out), a.M, a.N, a.K, a.x_rs, a.out_rs, tiles_m, grid, norm);
}

template <typename T>
static void run_mid_norm_t(const LinearArgs &a, int kind, const NormExchange &norm) {
    switch (kind) {
        case 11: launch_mid_norm<T, Mid64x64>(a, norm); break;
        case 15: launch_mid_norm<T, Mid128x64>(a, norm); break;
        case 17: launch_mid_norm<T, Mid128x128>(a, norm); break;
        case 18: launch_mid_norm<T, Mid192x128>(a, norm); break;
        case 19: launch_mid_norm<T, Mid192x192>(a, norm); break;
        case 20: launch_mid_norm<T, Mid128x256>(a, norm); break;
        case 22: launch_mid_norm<T, Mid192x96>(a, norm); break;
        default: launch_mid_norm<T, Mid256x128>(a, norm); break;
    }
}

void run_mid_norm(const LinearArgs &a, int dtype, int kind, const NormExchange &norm) {
    if (dtype == KERNL_F16) run_mid_norm_t<f16>(a, kind, norm);
    else run_mid_norm_t<bf16>(a, kind, norm);
}

}  // namespace kernl
