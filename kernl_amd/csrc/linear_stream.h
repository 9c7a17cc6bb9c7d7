// Linear layer for up to four rows of x (decoding steps of one sequence or a few): the weight is streamed past the caches in whole lines.
//
// What bounds it is the weight stream.  linear_skinny_kernel reads 16 weight rows in pieces of 128 bytes, two 16-byte loads a lane that each take half of every
// line, because that is how v_mfma_f32_16x16x32 wants its operand.  v_mfma_f32_4x4x4_16b takes 16 blocks of 4 weight rows x 4 k x 4 rows of x:
// with the blocks along k, lane l holds 16 bytes of weight row l % 4 at k = 8 (l / 4), so that one load of a wave is four runs of 256 contiguous bytes and two
// matrix instructions multiply all of it by four rows of x; the blocks' sums are added once at the end.  Whole lines can be read with a
// non-temporal hint (half lines cannot: the second half would be fetched again, a decoding step of four layers 400 -> 428 us).
// x (times the norm's weight) lies in LDS.  `ks` waves share a unit of rows and take batches of its k-steps by turns.
//
// us, linear_skinny_kernel -> this one, weights from HBM, fp16, one row / four rows of x: 12288 x 4096 rotated behind a norm 24.2 -> 19.3 / 26.8 -> 20.9,
// 32000 x 4096 behind a norm 49.5 -> 44.7 (5.9 TB/s) / 59.4 -> 46.2, 11008 x 4096 gated 36.6 -> 33.6 / 40.5 -> 35.8, 5120 x 5120 16.7 -> 12.5 / 18.0 -> 17.5,
// 4096 x 11008 20.4 -> 18.4 (one row), 4096 x 4096 9.0 -> 8.8 / 9.2 -> 8.9.  A decoding step of four such layers 400 -> 359.
#pragma once

#include "linear_kernels.h"

namespace kernl {

template <typename T>
struct Vec4x4 {
    typedef _Float16 type __attribute__((ext_vector_type(4)));
};
template <>
struct Vec4x4<bf16> {
    typedef short type __attribute__((ext_vector_type(4)));
};
__device__ __forceinline__ f32x4_acc mfma4(Vec4x4<f16>::type a, Vec4x4<f16>::type b, f32x4_acc c) { return __builtin_amdgcn_mfma_f32_4x4x4f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4_acc mfma4(Vec4x4<bf16>::type a, Vec4x4<bf16>::type b, f32x4_acc c) {
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a, b, c, 0, 0, 0);
}

constexpr int kStreamPlain = 0, kStreamGated = 1, kStreamRope = 2;
constexpr int kStreamWaves = 4, kStreamRows = 4, kStreamStep = 128;  // waves of a workgroup, most rows of x, k-values of one load
constexpr int kStreamLds = 48 * 1024;                                // most bytes of x in LDS (three workgroups a CU)
// bytes between rows of x in LDS: neighbouring rows start 16 banks apart
__host__ __device__ constexpr int stream_row_bytes(int K) { return 2 * K + 64; }

// G: groups of four weight rows of a wave (gate and value rows, the two members of rotated pairs, or neighbours)
template <typename T, int MODE, int G, bool RMS>
__global__ void __launch_bounds__(64 * kStreamWaves)
linear_stream_kernel(const T *__restrict__ X, const T *__restrict__ W, const T *__restrict__ bias, T *__restrict__ out, T *__restrict__ act_in, int M, int N,
                     int K, int64_t ldx, int64_t out_rs, int64_t out_cs, int64_t ai_rs, int64_t ai_cs, int act, const T *__restrict__ rms_w, float eps,
                     int ks, const SkinnyExtra ex) {
    static_assert(MODE == kStreamPlain || G == 2, "gates and values, pairs");
    typedef typename Vec8<T>::type vec8;
    typedef typename Vec4x4<T>::type vec4;
    constexpr bool ROPE = MODE == kStreamRope;
    constexpr int WAVES = kStreamWaves, ROWS = kStreamRows, THREADS = 64 * WAVES;
    constexpr int U = G == 1 ? 4 : 2;  // steps requested together: 4 KB a wave, two such batches in flight (8 KB each: no difference)
    constexpr int GO = MODE == kStreamGated ? 1 : G;  // groups of output columns
    extern __shared__ __attribute__((aligned(16))) unsigned char staged[];
    __shared__ float red_sq[RMS ? WAVES : 1][ROWS];
    __shared__ f32x4_acc red[WAVES][G][ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_k = wave % ks, unit = (int)blockIdx.x * (WAVES / ks) + wave / ks;
    // first output column of the unit, the weight rows of its groups, and the columns between two groups
    const int quads = ROPE ? ex.half / 4 : 1;
    const int n0 = ROPE ? unit / quads * (2 * ex.half) + unit % quads * 4 : unit * (4 * GO);
    const int apart = ROPE ? ex.half : MODE == kStreamGated ? 32 : 4;
    const int row0 = MODE == kStreamGated ? (n0 >> 5) * 64 + (n0 & 31) : n0, rows = MODE == kStreamGated ? 2 * N : N;
    const bool mine = n0 < N;
    const int steps = K / kStreamStep, batches = (steps + U - 1) / U;
    constexpr uint32_t kOutOfRange = 0x80000000u;
    const uint32_t off = (uint32_t)((lane & 3) * K * 2 + (lane >> 2) * 16);
    __amdgpu_buffer_rsrc_t rsrc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int row = row0 + apart * g, have = mine ? min(4, rows - row) : 0;
        rsrc[g] = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(W + (int64_t)(have > 0 ? row : 0) * K), 0, have > 0 ? have * K * 2 : 0, 0x00020000);
    }
    // Units start at different batches: rows a power of two apart would all ask the same memory channels at the same time (4096 x 11008
    // 19.8 -> 18.4 us)
    const int rot = (int)((unsigned)unit * 5u % (unsigned)batches);
    auto turned = [&](int b) __attribute__((always_inline)) { return b + rot >= batches ? b + rot - batches : b + rot; };
    u32x4 wf[2][U][G];
    auto request = [&](int buf, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = turned(b) * U + u;  // (past the end: out of range, no access; a branch would cost the compiler its count of loads in flight)
            const uint32_t at = b < batches && s < steps ? off : kOutOfRange;
#pragma unroll
            for (int g = 0; g < G; ++g) wf[buf][u][g] = __builtin_amdgcn_raw_buffer_load_b128(rsrc[g], at, s * (kStreamStep * 2), 2);  // 2: non-temporal
        }
    };
    f32x4_acc acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};
    const int m_lane = min(lane & 3, M - 1), stride = stream_row_bytes(K), x_at = m_lane * stride + (lane >> 2) * 16;
    auto multiply = [&](int buf, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = turned(b) * U + u;
            if (b >= batches || s >= steps) continue;
            const u32x4 xv = *reinterpret_cast<const u32x4 *>(staged + x_at + s * (kStreamStep * 2));
            const vec4 x0 = __builtin_bit_cast(vec4, u32x2{xv[0], xv[1]}), x1 = __builtin_bit_cast(vec4, u32x2{xv[2], xv[3]});
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const u32x4 w = wf[buf][u][g];
                acc[g] = mfma4(__builtin_bit_cast(vec4, u32x2{w[0], w[1]}), x0, acc[g]);
                acc[g] = mfma4(__builtin_bit_cast(vec4, u32x2{w[2], w[3]}), x1, acc[g]);
            }
        }
    };
    // What the epilogue needs from memory, requested first: lane j finishes row j of x.  Kept as it lies in memory and clamped instead of skipped: a
    // conversion or a branch here would wait for every load by itself (12288 x 4096 rotated 21.5 -> 19.3 us).
    const bool finishes = wave_k == 0 && mine && lane < M;
    uint32_t pre_bias[G][4], pre_res[GO][4];
    u32x4 c_tab[ROPE ? G : 1], s_tab[ROPE ? G : 1];
    const bool turns = ROPE && n0 < ex.rope_cols;  // (rope_cols is a multiple of the head size)
    if (finishes) {
        if (bias != nullptr)
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) pre_bias[g][i] = reinterpret_cast<const uint16_t *>(bias)[min(row0 + apart * g + i, rows - 1)];
        if (ex.residual != nullptr)
#pragma unroll
            for (int g = 0; g < GO; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    pre_res[g][i] = static_cast<const uint16_t *>(ex.residual)[m_lane * ex.res_rs + min(n0 + apart * g + i, N - 1) * ex.res_cs];
        if (turns) {
            auto entries = [&](const void *base, int64_t at) __attribute__((always_inline)) {  // four: 8 bytes of 16-bit values, or 16
                u32x4 raw = {0, 0, 0, 0};
                if (ex.table_dtype == KERNL_F32) {
                    __builtin_memcpy(&raw, static_cast<const float *>(base) + at, 16);
                } else {
                    u32x2 half;
                    __builtin_memcpy(&half, static_cast<const uint16_t *>(base) + at, 8);
                    raw[0] = half[0], raw[1] = half[1];
                }
                return raw;
            };
            const int64_t at = (int64_t)(m_lane / ex.rows_per_batch) * ex.t_bs + (int64_t)(m_lane % ex.rows_per_batch) * ex.t_ss + n0 % (2 * ex.half);
#pragma unroll
            for (int g = 0; g < (ROPE ? G : 0); ++g) {
                c_tab[g] = entries(ex.cos, at + apart * g);
                s_tab[g] = entries(ex.sin, at + apart * g);
            }
        }
    }
    // x to LDS, two 16-byte pieces of every row a thread and round; the first weights are requested behind the last of x
    {
        const int pieces = K / 8, rounds = (pieces + 2 * THREADS - 1) / (2 * THREADS);
        vec8 px[2][ROWS], pg[2];
        float squares[ROWS] = {};
        auto fetch = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int p = min((2 * t + i) * THREADS + tid, pieces - 1);
                if constexpr (RMS) pg[i] = *reinterpret_cast<const vec8 *>(rms_w + p * 8);
#pragma unroll
                for (int m = 0; m < ROWS; ++m)
                    if (m < M) px[i][m] = *reinterpret_cast<const vec8 *>(X + m * ldx + p * 8);
            }
        };
        auto stage = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int p = (2 * t + i) * THREADS + tid;
                if (p >= pieces) continue;
#pragma unroll
                for (int m = 0; m < ROWS; ++m) {
                    if (m >= M) continue;
                    if constexpr (RMS) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float v = to_float(px[i][m][e]);
                            squares[m] = fmaf(v, v, squares[m]);
                        }
                        px[i][m] = px[i][m] * pg[i];
                    }
                    *reinterpret_cast<vec8 *>(staged + m * stride + p * 16) = px[i][m];
                }
            }
        };
        fetch(0);
        for (int t = 1; t < rounds; ++t) {
            stage(t - 1);
            fetch(t);
        }
        request(0, wave_k);
        stage(rounds - 1);
        if constexpr (RMS)
#pragma unroll
            for (int m = 0; m < ROWS; ++m)
                if (m < M) {
                    const float sum = wave_sum(squares[m]);
                    if (lane == 0) red_sq[wave][m] = sum;
                }
    }
    __syncthreads();
    for (int b = wave_k; b < batches; b += 2 * ks) {
        request(1, b + ks);
        multiply(0, b);
        request(0, b + 2 * ks);
        multiply(1, b + ks);
    }
    // the 16 blocks' sums, then those of the waves that share the unit
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v = acc[g][i];
            v += dpp_mov<0x124>(v);  // row_ror:4
            v += dpp_mov<0x128>(v);  // row_ror:8
            acc[g][i] = rows4_sum(v);
        }
        if (ks > 1 && lane < ROWS) red[wave][g][lane] = acc[g];
    }
    if (ks > 1) __syncthreads();
    if (!finishes) return;
    float rstd = 1.0f;
    if constexpr (RMS) {
        float t = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) t += red_sq[w][lane];
        rstd = 1.0f / sqrtf(t / (float)K + eps);
    }
    float v[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        f32x4_acc sum = acc[g];
        for (int w = 1; w < ks; ++w) sum += red[wave + w][g][lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[g][i] = fmaf(sum[i], rstd, bias != nullptr ? to_float(__builtin_bit_cast(T, (uint16_t)pre_bias[g][i])) : 0.0f);
    }
    auto table = [&](const u32x4 &raw, int i) __attribute__((always_inline)) {
        const uint32_t word = raw[i], pair = raw[i >> 1];
        if (ex.table_dtype == KERNL_F32) return __builtin_bit_cast(float, word);
        const uint16_t half = (uint16_t)(pair >> (16 * (i & 1)));
        return ex.table_dtype == KERNL_F16 ? (float)__builtin_bit_cast(f16, half) : to_float(__builtin_bit_cast(bf16, half));
    };
#pragma unroll
    for (int g = 0; g < GO; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + apart * g + i;
            if (n >= N) continue;
            float y = v[g][i];
            if constexpr (ROPE) {
                if (turns) y = fmaf(y, table(c_tab[g], i), (g == 0 ? -v[1][i] : v[0][i]) * table(s_tab[g], i));
            } else {
                if (MODE == kStreamPlain && act_in != nullptr) act_in[lane * ai_rs + n * ai_cs] = from_float<T>(y);
                y = apply_act16(y, act);
                if (MODE == kStreamGated) y *= v[G - 1][i];
            }
            if (ex.residual != nullptr) y += to_float(__builtin_bit_cast(T, (uint16_t)pre_res[g][i]));
            out[lane * out_rs + n * out_cs] = from_float<T>(y);
        }
}

// Waves that share a unit of rows: the fewest that give every CU nearly as many workgroups as the fullest one has (12288 x 4096 rotated, 1536 units: one wave 22.3 us,
// two 19.4, four 20.7), else the most that still run at the same time (11008 x 4096 gated, 2752 units: 33.9, 32.5, 35.3); 32000 x 4096, 4000 units: 44.6, 45.8, 48.1.
static int stream_split(int64_t units) {
    int most = 1;
    for (int ks = 1; ks <= kStreamWaves; ks *= 2) {
        const int64_t groups = (units * ks + kStreamWaves - 1) / kStreamWaves, rounds = (groups + 255) / 256;
        if (ks > 1 && groups > 6 * 256) break;
        most = ks;
        if ((double)groups >= 0.95 * 256.0 * (double)rounds) break;
    }
    return most;
}

// Whether a linear layer of up to 64 rows runs on it: at most four rows of x, which fit LDS beside those of other workgroups (us, linear_skinny_kernel / this one: four
// rows of 4096 x 11008 22.1 / 24.3, eight of 4096 rotated 28.8 / 31.1), and a K that is worth the staging (one row of 768 x 3072 6.0 / 4.7, 513 x 1536 4.4 / 3.9,
// 2048 x 2048 5.1 / 4.7, but 1024 x 1024 4.0 / 4.0, 768 x 768 3.7 / 4.0, 3072 x 768 3.8 / 4.9).
static bool stream_takes(const LinearArgs &a) {
    return a.M <= kStreamRows && a.K % kStreamStep == 0 && a.K >= 1536 && a.M * (int64_t)stream_row_bytes(a.K) <= kStreamLds && (int64_t)a.N * a.K >= (1 << 19);
}

template <typename T, int MODE, int G, bool RMS>
static void launch_stream_kernel(const LinearArgs &a, const void *rms_w, float eps, const SkinnyExtra &ex) {
    const int n_out = MODE == kStreamGated ? a.N / 2 : a.N, per_unit = MODE == kStreamGated ? 4 : 4 * G;
    const int64_t units = (n_out + per_unit - 1) / per_unit;
    const int ks = stream_split(units);
    hipLaunchKernelGGL((linear_stream_kernel<T, MODE, G, RMS>), dim3((unsigned)((units * ks + kStreamWaves - 1) / kStreamWaves)), dim3(64 * kStreamWaves),
                       a.M * stream_row_bytes(a.K), a.st, static_cast<const T *>(a.x), static_cast<const T *>(a.w), static_cast<const T *>(a.bias),
                       static_cast<T *>(a.out), static_cast<T *>(a.act_in), a.M, n_out, a.K, a.x_rs, a.out_rs, a.out_cs, a.ai_rs, a.ai_cs,
                       a.act & (kGluBit - 1), static_cast<const T *>(rms_w), eps, ks, ex);
}

// The linear layer, gated (a.act) or with rotated columns (ex.half), behind an RMSNorm (rms_w) or not.
template <typename T>
static void launch_stream(const LinearArgs &a, const void *rms_w, float eps, const SkinnyExtra &ex) {
    auto by_norm = [&](auto mode_c, auto g_c) {
        constexpr int MODE = decltype(mode_c)::value, G = decltype(g_c)::value;
        if (rms_w != nullptr) launch_stream_kernel<T, MODE, G, true>(a, rms_w, eps, ex);
        else launch_stream_kernel<T, MODE, G, false>(a, rms_w, eps, ex);
    };
    if (ex.half > 0) launch_stream_kernel<T, kStreamRope, 2, true>(a, rms_w, eps, ex);  // (always behind a norm)
    else if (a.act & kGluBit) by_norm(IntC<kStreamGated>(), IntC<2>());
    else if (a.N >= 8192) by_norm(IntC<kStreamPlain>(), IntC<2>());
    else by_norm(IntC<kStreamPlain>(), IntC<1>());
}

}  // namespace kernl
