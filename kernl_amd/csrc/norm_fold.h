// LayerNorm between two linear layers without a kernel of its own ("deferred" norm): the layer in front stores the
// UN-normalised rows s = round(x W^T + b + residual) together with per-row statistics, the layer behind multiplies s by the
// weight with gamma folded in and normalises its fp32 sums,
//     LN(s) W^T + b  =  rstd (s (W gamma)^T - mean colsum) + (b + W beta),     colsum[n] = sum_k (W gamma)[n][k],
// and where LN(s) itself is needed again — as the residual of the next addition — it is computed from s on the fly, in
// fp32.  One rounding of s takes the place of the rounding of LN(s); no operand gains one.
//
// Statistics of a row: for every 32 columns the pair (sum, sum of squared deviations from their mean) of the stored
// 16-bit values, fp32, row-major [rows][columns / 32].  Groups are merged around the first group's mean, so a mean far
// from zero costs no accuracy.
#pragma once

#include "common.h"

namespace kernl {

constexpr int kNormGroup = 32;       // columns per statistics pair
constexpr int kNormMaxGroups = 32;   // widths up to 1024

// MODE of the kernels that take part
constexpr int kNormNone = 0;    // plain epilogue
constexpr int kNormApply = 1;   // x is un-normalised: fold its norm into the epilogue
constexpr int kNormAdd = 2;     // add a residual (itself normalised on the fly when it has statistics), store statistics

struct NormFold {
    const float *in_stats = nullptr;   // kNormApply: of x; kNormAdd: of the residual, or null
    int in_groups = 0;                 // statistics pairs per row of in_stats
    float eps = 0.0f;
    const float *colsum = nullptr;     // kNormApply, [N]
    const float *bias32 = nullptr;     // kNormApply, [N]
    const void *residual = nullptr;    // kNormAdd, [M, N] 16-bit rows
    int64_t res_rs = 0;
    const void *gamma = nullptr, *beta = nullptr;  // kNormAdd with in_stats: of the residual's norm; beta may be null
    float *out_stats = nullptr;        // kNormAdd, [M, N / 32] pairs
};

// Running merge of a row's statistics pairs: deviations d of the groups' means from a pivot (any of them).
struct NormMerge {
    float d = 0.0f, dd = 0.0f, m2 = 0.0f;
    __device__ __forceinline__ void take(const f32x2 pair, float pivot) {
        const float e = fmaf(pair[0], 1.0f / kNormGroup, -pivot);
        d += e;
        dd = fmaf(e, e, dd);
        m2 += pair[1];
    }
    __device__ __forceinline__ void finish(float pivot, int groups, float eps, float &mean, float &rstd) const {
        const float inv = 1.0f / (float)groups, dm = d * inv;
        mean = pivot + dm;
        const float var = fmaf(m2, inv * (1.0f / kNormGroup), fmaxf(fmaf(-dm, dm, dd * inv), 0.0f));
        rstd = rsqrtf(var + eps);
    }
};

// sum over the eight lanes 8 i .. 8 i + 7, to each of them
__device__ __forceinline__ float oct_sum(float v) {
    v += dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_mov<0x141>(v);  // row_half_mirror
    return v;
}

// four consecutive 16-bit values as floats
template <typename T>
__device__ __forceinline__ void unpack4(u32x2 raw, float (&dst)[4]) {
    typedef T pair_t __attribute__((ext_vector_type(2)));
    const uint32_t r0 = raw[0], r1 = raw[1];  // (a bit cast straight from a vector ELEMENT reads the vector's first one)
    const pair_t lo = __builtin_bit_cast(pair_t, r0), hi = __builtin_bit_cast(pair_t, r1);
    dst[0] = to_float(lo[0]); dst[1] = to_float(lo[1]); dst[2] = to_float(hi[0]); dst[3] = to_float(hi[1]);
}

}  // namespace kernl
