// Launchers of the wide kernels with dealt k-tiles (see linear_kernels.h): a translation unit, and with it a code object, of its own.
// Among them, the same instructions of the forms without dealt k-tiles lie elsewhere in theirs and run 0.7 % slower (16384 x 768 x 3072
// with residual 71.0 -> 71.3 us, 16384 x 2304 x 768 58.9 -> 59.3: 80 KB of code a kernel against 64 KB of instruction cache).
#include "linear_kernels.h"

namespace kernl {

bool run_wide_dealt_takes(const LinearArgs &a) {
    const bool plain = a.act == KERNL_ACT_NONE, silu_gates = a.act == (kGluBit | KERNL_ACT_SILU);
    return (plain || silu_gates) && k_tiles_dealt(a.N, a.K) && a.K % 256 == 0;
}

template <typename T, int NBN>
static void launch_wide_dealt(const LinearArgs &a) {
    if constexpr (NBN == 8) {
        if (a.act & kGluBit) {
            if (a.row_scale != nullptr) launch_wide_act<T, kGluBit | KERNL_ACT_SILU, 8, false, true, false, true>(a);
            else launch_wide_act<T, kGluBit | KERNL_ACT_SILU, 8, false, false, false, true>(a);
            return;
        }
    }
    if (a.residual != nullptr) launch_wide_act<T, KERNL_ACT_NONE, NBN, false, false, true, true>(a);
    else if (a.row_scale != nullptr) launch_wide_act<T, KERNL_ACT_NONE, NBN, false, true, false, true>(a);
    else launch_wide_act<T, KERNL_ACT_NONE, NBN, false, false, false, true>(a);
}

template <typename T, int NBN>
static void launch_wide_half_dealt(const LinearArgs &a) {
    if (a.residual != nullptr) launch_wide_half_act<T, KERNL_ACT_NONE, NBN, false, false, true, true>(a);
    else if (a.row_scale != nullptr) launch_wide_half_act<T, KERNL_ACT_NONE, NBN, false, true, false, true>(a);
    else launch_wide_half_act<T, KERNL_ACT_NONE, NBN, false, false, false, true>(a);
}

void run_wide_dealt(const LinearArgs &a, int dtype, int cols) {
    if (dtype == KERNL_F16) cols == 192 ? launch_wide_dealt<f16, 6>(a) : launch_wide_dealt<f16, 8>(a);
    else cols == 192 ? launch_wide_dealt<bf16, 6>(a) : launch_wide_dealt<bf16, 8>(a);
}

void run_wide_half_dealt(const LinearArgs &a, int dtype, int cols) {
    if (dtype == KERNL_F16) cols == 192 ? launch_wide_half_dealt<f16, 6>(a) : launch_wide_half_dealt<f16, 8>(a);
    else cols == 192 ? launch_wide_half_dealt<bf16, 6>(a) : launch_wide_half_dealt<bf16, 8>(a);
}

}  // namespace kernl
