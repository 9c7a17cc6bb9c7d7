// What follows a product whose K was split (linear_mid.hip): the ranges' fp32 sums [splits][M][part_rs] are added in order, and the
// launch that has to read them anyway finishes the row — bias and activation; the residual with the row statistics of an
// RMSNorm; the residual and the whole LayerNorm — so that an encoder's add + LayerNorm launch or a prompt's add + statistics launch
// is this one.
//
// Bound by launch and one trip to memory (the sums lie in the memory-side cache).  Rows are kept in registers: a workgroup per row, or
// a wave where there are rows enough of up to 1024 columns.
#include "linear_kernels.h"
#include "norm_fold.h"

namespace kernl {

// Four columns in each of CH chunks of a row, `step` columns apart: the ranges' sums, added in order.  All loads are requested before the first
// addition, which takes the number of ranges as a constant: a branch per range in front of each load costs a wait each (231 x 768, five
// ranges: 9.8 us).
template <int S, int CH>
__device__ __forceinline__ void split_sums_of(const float *__restrict__ p, int64_t range_stride, int step, int n, int N, f32x4_acc (&sum)[CH]) {
    f32x4_acc v[CH][S];
#pragma unroll
    for (int c = 0; c < CH; ++c)
        if (n + c * step < N)
#pragma unroll
            for (int s = 0; s < S; ++s) v[c][s] = *reinterpret_cast<const f32x4_acc *>(p + s * range_stride + n + c * step);
#pragma unroll
    for (int c = 0; c < CH; ++c)
        if (n + c * step < N) {
            sum[c] = v[c][0];
#pragma unroll
            for (int s = 1; s < S; ++s) sum[c] += v[c][s];
        }
}
template <int CH>
__device__ __forceinline__ void split_sums(const float *__restrict__ p, int splits, int64_t range_stride, int step, int n, int N, f32x4_acc (&sum)[CH]) {
    switch (splits) {
        case 2: split_sums_of<2, CH>(p, range_stride, step, n, N, sum); break;
        case 3: split_sums_of<3, CH>(p, range_stride, step, n, N, sum); break;
        case 4: split_sums_of<4, CH>(p, range_stride, step, n, N, sum); break;
        case 5: split_sums_of<5, CH>(p, range_stride, step, n, N, sum); break;
        case 6: split_sums_of<6, CH>(p, range_stride, step, n, N, sum); break;
        case 7: split_sums_of<7, CH>(p, range_stride, step, n, N, sum); break;
        default: split_sums_of<8, CH>(p, range_stride, step, n, N, sum); break;
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
split_finish_plain_kernel(const float *__restrict__ part, int splits, int64_t part_rs, const T *__restrict__ bias, T *__restrict__ out,
                          T *__restrict__ act_in, int M, int N, int64_t out_rs, int64_t out_cs, int64_t ai_rs, int64_t ai_cs, int act) {
    const int64_t chunks = part_rs / 4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)M * chunks) return;
    const int m = (int)(i / chunks), n = (int)(i % chunks) * 4;
    float b[4];
    load_bias4<T>(bias, n, N, ((uintptr_t)bias & 7) == 0, b);
    f32x4_acc sums[1];
    split_sums<1>(part + (int64_t)m * part_rs, splits, (int64_t)M * part_rs, 0, n, (int)part_rs, sums);
    const f32x4_acc sum = sums[0];
    float v[4], y[4];
    auto finish = [&](auto act_c) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = sum[e] + b[e];
            y[e] = apply_act16(v[e], decltype(act_c)::value);
        }
    };
    switch (act) {
        case KERNL_ACT_RELU: finish(IntC<KERNL_ACT_RELU>()); break;
        case KERNL_ACT_TANH: finish(IntC<KERNL_ACT_TANH>()); break;
        case KERNL_ACT_GELU_ERF: finish(IntC<KERNL_ACT_GELU_ERF>()); break;
        case KERNL_ACT_GELU_TANH: finish(IntC<KERNL_ACT_GELU_TANH>()); break;
        case KERNL_ACT_SILU: finish(IntC<KERNL_ACT_SILU>()); break;
        default: finish(IntC<KERNL_ACT_NONE>()); break;
    }
    auto store = [&](T *p, int64_t rs, int64_t cs, const float *w) __attribute__((always_inline)) {
        T *q = p + (int64_t)m * rs + (int64_t)n * cs;
        if (cs == 1 && n + 4 <= N && ((uintptr_t)q & 7) == 0) {
            *reinterpret_cast<u32x2 *>(q) = u32x2{pack2<T>(w[0], w[1]), pack2<T>(w[2], w[3])};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < N) q[e * cs] = from_float<T>(w[e]);
        }
    };
    store(out, out_rs, out_cs, y);
    if (act_in != nullptr) store(act_in, ai_rs, ai_cs, v);
}

// A row per group of WAVES waves, CH chunks of four columns per lane.  N % 4 == 0, out, residual, bias, gamma and beta 8-byte aligned.
template <typename T, int FINISH, int WAVES, int CH>
__global__ void __launch_bounds__(256)
split_finish_rows_kernel(const float *__restrict__ part, int splits, int64_t part_rs, const T *__restrict__ bias, const T *__restrict__ residual,
                         int64_t res_rs, const T *__restrict__ gamma, const T *__restrict__ beta, float eps, T *__restrict__ out, int64_t out_rs,
                         float *__restrict__ rstd_out, int M, int N) {
    constexpr int G = 64 * WAVES;
    __shared__ float red[2][4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, t = WAVES == 1 ? lane : (int)threadIdx.x;
    const int m = WAVES == 1 ? blockIdx.x * 4 + wave : blockIdx.x;
    if (WAVES == 1 && m >= M) return;  // (no barrier below in this form)
    auto row_sum = [&](float v, int slot) -> float {
        v = wave_sum(v);
        if (WAVES == 1) return v;
        if (lane == 0) red[slot][wave] = v;
        __syncthreads();
        return (red[slot][0] + red[slot][1]) + (red[slot][2] + red[slot][3]);
    };
    const float inv_n = 1.0f / (float)N;
    const float *p = part + (int64_t)m * part_rs;
    u32x2 rv[CH], bv[CH], gv[FINISH == kFinishLayerNorm ? CH : 1], ev[FINISH == kFinishLayerNorm ? CH : 1];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int n = (t + c * G) * 4;
        rv[c] = bv[c] = u32x2{0, 0};
        if (n >= N) continue;
        rv[c] = *reinterpret_cast<const u32x2 *>(residual + (int64_t)m * res_rs + n);
        if (bias != nullptr) bv[c] = *reinterpret_cast<const u32x2 *>(bias + n);
        if constexpr (FINISH == kFinishLayerNorm) {
            gv[c] = *reinterpret_cast<const u32x2 *>(gamma + n);
            ev[c] = beta != nullptr ? *reinterpret_cast<const u32x2 *>(beta + n) : u32x2{0, 0};
        }
    }
    f32x4_acc sums[CH];
    split_sums<CH>(p, splits, (int64_t)M * part_rs, G * 4, t * 4, N, sums);
    float y[CH][4], sum = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int n = (t + c * G) * 4;
        y[c][0] = y[c][1] = y[c][2] = y[c][3] = 0.0f;
        if (n >= N) continue;
        const f32x4_acc s = sums[c];
        float r[4], b[4];
        unpack4<T>(rv[c], r);
        unpack4<T>(bv[c], b);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (FINISH == kFinishLayerNorm) {
                y[c][e] = s[e] + b[e] + r[e];
                sum += y[c][e];
            } else {
                y[c][e] = to_float(from_float<T>(to_float(from_float<T>(s[e] + b[e])) + r[e]));
                sum = fmaf(y[c][e], y[c][e], sum);
            }
        }
    }
    float mean = 0.0f, rstd = 1.0f;
    if constexpr (FINISH == kFinishLayerNorm) {
        mean = row_sum(sum, 0) * inv_n;
        float dev = 0.0f;
#pragma unroll
        for (int c = 0; c < CH; ++c)
            if ((t + c * G) * 4 < N)
#pragma unroll
                for (int e = 0; e < 4; ++e) dev = fmaf(y[c][e] - mean, y[c][e] - mean, dev);
        rstd = rsqrtf(row_sum(dev, 1) * inv_n + eps);
    } else if constexpr (FINISH == kFinishRmsStats) {
        const float r = rsqrtf(row_sum(sum, 0) * inv_n + eps);
        if (t == 0) rstd_out[m] = r;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int n = (t + c * G) * 4;
        if (n >= N) continue;
        float z[4];
        if constexpr (FINISH == kFinishLayerNorm) {
            float ga[4], be[4];
            unpack4<T>(gv[c], ga);
            unpack4<T>(ev[c], be);
#pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = fmaf((y[c][e] - mean) * rstd, ga[e], be[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = y[c][e];
        }
        *reinterpret_cast<u32x2 *>(out + (int64_t)m * out_rs + n) = u32x2{pack2<T>(z[0], z[1]), pack2<T>(z[2], z[3])};
    }
}

template <typename T, int FINISH>
static void launch_rows(const LinearArgs &a, const MidSplit &s, const SplitFinish &f) {
    auto go = [&](auto kern, int rows_per_block) {
        hipLaunchKernelGGL(kern, dim3((unsigned)((a.M + rows_per_block - 1) / rows_per_block)), dim3(256), 0, a.st, s.part, s.splits, s.part_rs,
                           static_cast<const T *>(a.bias), static_cast<const T *>(a.residual), a.res_rs, static_cast<const T *>(f.gamma),
                           static_cast<const T *>(f.beta), f.eps, static_cast<T *>(a.out), a.out_rs, f.rstd, a.M, a.N);
    };
    if (a.N <= 1024 && a.M <= 1024) go(split_finish_rows_kernel<T, FINISH, 4, 1>, 1);
    else if (a.N <= 768) go(split_finish_rows_kernel<T, FINISH, 1, 3>, 4);
    else if (a.N <= 1024) go(split_finish_rows_kernel<T, FINISH, 1, 4>, 4);
    else if (a.N <= 4096) go(split_finish_rows_kernel<T, FINISH, 4, 4>, 1);
    else go(split_finish_rows_kernel<T, FINISH, 4, 8>, 1);
}

template <typename T>
static void run_split_finish_t(const LinearArgs &a, const MidSplit &s, const SplitFinish &f) {
    switch (f.kind) {
        case kFinishResidual: launch_rows<T, kFinishResidual>(a, s, f); break;
        case kFinishRmsStats: launch_rows<T, kFinishRmsStats>(a, s, f); break;
        case kFinishLayerNorm: launch_rows<T, kFinishLayerNorm>(a, s, f); break;
        default: {
            const int64_t work = (int64_t)a.M * (s.part_rs / 4);
            hipLaunchKernelGGL((split_finish_plain_kernel<T>), dim3((unsigned)((work + 255) / 256)), dim3(256), 0, a.st, s.part, s.splits, s.part_rs,
                               static_cast<const T *>(a.bias), static_cast<T *>(a.out), static_cast<T *>(a.act_in), a.M, a.N, a.out_rs,
                               a.out_cs, a.ai_rs, a.ai_cs, a.act);
        }
    }
}

void run_split_finish(const LinearArgs &a, int dtype, const MidSplit &split, const SplitFinish &finish) {
    if (dtype == KERNL_F16) run_split_finish_t<f16>(a, split, finish);
    else run_split_finish_t<bf16>(a, split, finish);
}

}  // namespace kernl
