// LayerNorm between two linear layers without a kernel of its own ("deferred" norm), for up to 64 rows: the layer in front
// stores the rows s = x W^T + b + residual in fp32, un-normalised, with statistics; the layer behind normalises them on
// their way into its matrix instructions,
//     LN(s) = (s - mean) rstd gamma + beta    in fp32, rounded once to the 16-bit operand,
// which is what a LayerNorm kernel would have stored, and where LN(s) is needed again — as the residual of the next
// addition — it is computed from s the same way and not rounded at all.  Against a linear kernel and an add + LayerNorm kernel two
// roundings are gone (the projection's and the residual's) and none is new, whatever the rows' mean and the norm's parameters
// are.  (An earlier form stored s in 16 bits and folded gamma into the weight: its error grew with mean / std of the rows.)
//
// More rows keep their LayerNorm kernel: a product in tiles of 64 rows and more is bound by its tile loads, and fp32 rows
// double those of x.
//
// Statistics of a row: for every 16 columns the pair (sum, sum of squared deviations from their mean) of the fp32 values,
// row-major [rows][groups].  Groups are merged around the first group's mean, so a mean far from zero costs no accuracy.
#pragma once

#include "common.h"

namespace kernl {

constexpr int kNormGroup = 16;       // columns per statistics pair
constexpr int kNormMaxRows = 64;     // rows that tiles of whole statistics groups are built for
constexpr int kNormMaxGroups = 64;   // widths up to 1024

// MODE of the kernels in front of a norm
constexpr int kNormNone = 0;    // plain epilogue
constexpr int kNormExchange = 1;  // add a 16-bit residual and normalise, the statistics exchanged with the other column tiles (norm_exchange.h)
constexpr int kNormAdd = 2;     // add a residual (itself normalised on the fly when it has statistics), store fp32 rows and statistics

struct NormFold {
    const float *in_stats = nullptr;   // of the residual (kNormAdd; may be null) or of x (the layer behind)
    int in_groups = 0;                 // statistics pairs per row of in_stats
    float inv_groups = 1.0f;
    float eps = 0.0f;
    const void *residual = nullptr;    // kNormAdd, [M, N]: fp32 rows with in_stats, 16-bit rows without
    int64_t res_rs = 0;
    const void *gamma = nullptr, *beta = nullptr;  // with in_stats: of that norm; beta may be null
    void stats_of(int64_t width) {     // in_stats describe rows of `width` columns
        in_groups = (int)(width / kNormGroup);
        inv_groups = 1.0f / (float)in_groups;
    }
    float *out_stats = nullptr;        // kNormAdd, [M, N / kNormGroup] pairs
};

// Running merge of a row's statistics pairs: deviations d of the groups' means from a pivot (any of them).
struct NormMerge {
    static constexpr float kInvGroup = 1.0f / kNormGroup;
    float d = 0.0f, dd = 0.0f, m2 = 0.0f;
    __device__ __forceinline__ void take(const f32x2 pair, float pivot) {
        const float e = fmaf(pair[0], kInvGroup, -pivot);
        d += e;
        dd = fmaf(e, e, dd);
        m2 += pair[1];
    }
    // (mean, 1 / std) of the row
    __device__ __forceinline__ f32x2 finish(float pivot, const NormFold &nf) const {
        const float dm = d * nf.inv_groups;
        const float var = fmaf(m2, nf.inv_groups * kInvGroup, fmaxf(fmaf(-dm, dm, dd * nf.inv_groups), 0.0f));
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
