// LayerNorm between two linear layers without a kernel of its own ("deferred" norm): the layer in front stores the
// UN-normalised rows s = round(x W^T + b + residual) together with per-row statistics, the layer behind multiplies s by the
// weight with gamma folded in and normalises its fp32 sums,
//     LN(s) W^T + b  =  rstd (s (W gamma)^T - mean colsum) + (b + W beta),     colsum[n] = sum_k (W gamma)[n][k],
// and where LN(s) itself is needed again — as the residual of the next addition — it is computed from s on the fly, in
// fp32.  One rounding of s takes the place of the rounding of LN(s); no operand gains one.
//
// Statistics of a row: for every 32 columns (16 up to 64 rows, whose tiles are that narrow) the pair (sum, sum of squared deviations from their mean) of the stored
// 16-bit values, fp32, row-major [rows][groups].  Groups are merged around the first group's mean, so a mean far
// from zero costs no accuracy.
#pragma once

#include "common.h"

namespace kernl {

constexpr int kNormGroup = 32;       // columns per statistics pair ...
constexpr int kNormGroupFew = 16;    // ... and of inputs of at most
constexpr int kNormFewRows = 64;     // so many rows
constexpr int kNormMaxGroups = 32;   // widths up to 1024
static inline int norm_group_of(int64_t rows) { return rows <= kNormFewRows ? kNormGroupFew : kNormGroup; }

// MODE of the kernels that take part
constexpr int kNormNone = 0;    // plain epilogue
constexpr int kNormApply = 1;   // x is un-normalised: fold its norm into the epilogue
constexpr int kNormAdd = 2;     // add a residual (itself normalised on the fly when it has statistics), store statistics

struct NormFold {
    const float *in_stats = nullptr;   // kNormApply: of x; kNormAdd: of the residual, or null
    int in_groups = 0;                 // statistics pairs per row of in_stats
    int group = kNormGroup;            // columns of a pair
    float inv_group = 1.0f / kNormGroup, inv_groups = 1.0f;
    float eps = 0.0f;
    const float *colsum = nullptr;     // kNormApply, [N]
    const float *bias32 = nullptr;     // kNormApply, [N]
    const void *residual = nullptr;    // kNormAdd, [M, N] 16-bit rows
    int64_t res_rs = 0;
    const void *gamma = nullptr, *beta = nullptr;  // kNormAdd with in_stats: of the residual's norm; beta may be null
    void stats_of(int64_t rows, int64_t width) {  // in_stats describe `rows` rows of `width` columns
        group = norm_group_of(rows);
        in_groups = (int)(width / group);
        inv_group = 1.0f / (float)group;
        inv_groups = 1.0f / (float)in_groups;
    }
    float *out_stats = nullptr;        // kNormAdd, [M, N / group] pairs
};

// Running merge of a row's statistics pairs: deviations d of the groups' means from a pivot (any of them).
struct NormMerge {
    float d = 0.0f, dd = 0.0f, m2 = 0.0f;
    __device__ __forceinline__ void take(const f32x2 pair, float pivot, float inv_group) {
        const float e = fmaf(pair[0], inv_group, -pivot);
        d += e;
        dd = fmaf(e, e, dd);
        m2 += pair[1];
    }
    // (mean, 1 / std) of the row
    __device__ __forceinline__ f32x2 finish(float pivot, const NormFold &nf) const {
        const float dm = d * nf.inv_groups;
        const float var = fmaf(m2, nf.inv_groups * nf.inv_group, fmaxf(fmaf(-dm, dm, dd * nf.inv_groups), 0.0f));
        return f32x2{pivot + dm, rsqrtf(var + nf.eps)};
    }
};

// sum over the eight (four) lanes that share lane / 8 (lane / 4), to each of them
__device__ __forceinline__ float quad_sum(float v) {
    v += dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
    return v;
}
__device__ __forceinline__ float oct_sum(float v) {
    v = quad_sum(v);
    v += dpp_mov<0x141>(v);  // row_half_mirror
    return v;
}

// four consecutive 16-bit values as floats
template <typename T>
__device__ __forceinline__ void unpack4(u32x2 raw, float *dst) {
    typedef T pair_t __attribute__((ext_vector_type(2)));
    const uint32_t r0 = raw[0], r1 = raw[1];  // (a bit cast straight from a vector ELEMENT reads the vector's first one)
    const pair_t lo = __builtin_bit_cast(pair_t, r0), hi = __builtin_bit_cast(pair_t, r1);
    dst[0] = to_float(lo[0]); dst[1] = to_float(lo[1]); dst[2] = to_float(hi[0]); dst[3] = to_float(hi[1]);
}

// bias[n .. n + 3] as floats (zeros past N or without a bias): one 8-byte load where the four are inside and aligned
template <typename T>
__device__ __forceinline__ void load_bias4(const T *__restrict__ bias, int n, int N, bool vec_ok, float (&dst)[4]) {
    if (bias != nullptr && vec_ok && n + 4 <= N) {
        unpack4<T>(*reinterpret_cast<const u32x2 *>(bias + n), dst);
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = (bias != nullptr && n + e < N) ? to_float(bias[n + e]) : 0.0f;
}

}  // namespace kernl
