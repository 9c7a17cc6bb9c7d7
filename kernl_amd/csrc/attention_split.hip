// Causal flash attention for grids too small for 128-row workgroups that walk all keys alone: a prompt, some heads of a few hundred to
// a few thousand rows, new rows over a cache; no mask.
//
// What bounds such a launch is the chain of key tiles: with one 128-row workgroup a CU, a SIMD holds one wave and a tile of 128 keys takes
// 2.2 us (head size 128) of which the matrix cores work 0.85.  Here a workgroup has eight waves, two groups of 32 rows times four groups
// of 32 keys that share every key tile of 128 (one double buffer, one barrier a tile): half the rows and a quarter of the keys for each
// wave, two waves on every SIMD, and the longest workgroups go first.  The key groups' results — reference, row sum, accumulator — meet
// in LDS at the end, where each wave finishes its share of the features.  Graph replay, us, [heads, rows, head size], streaming or
// pipelined kernel -> this one: [16,333,128] 10.9 -> 9.6, [16,700,128] 15.7 -> 14.0, [16,1111,128] 21.2 -> 18.4, [12,1500,128] 28.7 ->
// 23.2, [8,2048,128] 32.5 -> 28.9, [12,512,64] 9.9 -> 8.1, [12,900,64] 14.4 -> 11.1.  Four groups of 32 rows times two of keys: 5 to 25 %
// behind this shape; without causality the pipelined kernel is ahead of both.
//
// The softmax keeps a reference per row that moves (with a rescale of the accumulator) when a score exceeds it by more than 2^8; whether
// any does is a vote of the wave, so the maximum crosses lanes only then.  Operand layout as in attention_short.hip: lane (r, g)
// ends the score products with keys 16 n + 4 g .. + 3 of query r, and the value products use that order of keys.
#include "attention_common.h"

namespace kernl {

// maximum / sum over the four lanes that share lane % 16, to each of them
__device__ __forceinline__ float quarters_max(float v) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, v);
    const auto s = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    return halves32_max(fmaxf(__builtin_bit_cast(float, (uint32_t)s[0]), __builtin_bit_cast(float, (uint32_t)s[1])));
}
__device__ __forceinline__ float quarters_sum(float v) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, v);
    const auto s = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    return halves32_sum(__builtin_bit_cast(float, (uint32_t)s[0]) + __builtin_bit_cast(float, (uint32_t)s[1]));
}

template <typename T, int D>
__global__ void __launch_bounds__(512, 2) attention_split_kernel(const AttnParams p) {
    typedef typename Vec8<T>::type vec8;
    constexpr int QG = 2, KG = 8 / QG, BM = 32 * QG, BN = 128, KW = BN / KG;         // key groups, rows, keys a tile, keys of a wave
    constexpr int KS = D / 32, FB = D / 16, ROW = D * 2, CPR = D / 8, NB = KW / 16;
    constexpr int TILE = BN * ROW, STAGE = 2 * TILE;                          // keys, values
    constexpr int LOADS = TILE / 8192, ROWS = 64 / CPR;                       // 1 KB loads of a wave for keys (values); rows of a load
    extern __shared__ __attribute__((aligned(16))) unsigned char tiles[];    // two stages; the accumulators at the end
    __shared__ float ref_of[8][32], sum_of[8][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int qg = wave % QG, kg = wave / QG;
    const int heads = p.B * p.H, bh = (int)blockIdx.x % heads, rank = (int)blockIdx.x / heads, b = bh / p.H, h = bh % p.H;
    const int qt = p.nq_tiles - 1 - rank;  // the longest first
    const int M = p.M, N = p.N, m0 = qt * BM + qg * 32;
    const int n_end = min(N, qt * BM + BM + p.causal_off), n_tiles = (n_end + BN - 1) / BN;

    const T *qp = static_cast<const T *>(p.q) + b * p.qs[0] + h * p.qs[1];
    vec8 qf[2][KS];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const T *qrow = qp + (int64_t)min(m0 + 16 * i + r, M - 1) * p.qs[2];
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[i][s] = *reinterpret_cast<const vec8 *>(qrow + 32 * s + 8 * g);
    }
    // tile loads, straight into LDS: load i of a wave fills rows (8 i + wave) * ROWS ..; rows past the last key lie outside the buffer
    // and arrive as zeros.  Keys swizzled for whole-row fragment reads, values by value_flip.
    typedef __attribute__((address_space(3))) void lds_void;
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_void *)tiles;
    const uint32_t k_step = (uint32_t)p.ks[2] * 2, v_step = (uint32_t)p.vs[2] * 2;
    const uint64_t ka = (uint64_t)(uintptr_t)(static_cast<const T *>(p.k) + b * p.ks[0] + h * p.ks[1]);
    const uint64_t va = (uint64_t)(uintptr_t)(static_cast<const T *>(p.v) + b * p.vs[0] + h * p.vs[1]);
    const u32x4 krsrc = {(uint32_t)ka, (uint32_t)(ka >> 32) & 0xFFFFu, (N - 1) * k_step + D * 2, 0x00020000u};
    const u32x4 vrsrc = {(uint32_t)va, (uint32_t)(va >> 32) & 0xFFFFu, (N - 1) * v_step + D * 2, 0x00020000u};
    uint32_t k_at[LOADS], v_at[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (8 * i + wave) * ROWS + lane / CPR, c = lane % CPR;
        k_at[i] = row * k_step + swz_chunk<ROW>(row, c) * 16;
        v_at[i] = row * v_step + (c ^ value_flip<D>(row)) * 16;
    }
    auto request = [&](int tile, int stage) __attribute__((always_inline)) {
        const uint32_t at = lds + stage * STAGE + wave * 1024;
        const uint32_t ko = (uint32_t)tile * BN * k_step, vo = (uint32_t)tile * BN * v_step;
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(at + i * 8192), "v"(k_at[i]), "s"(krsrc), "s"(ko) : "memory", "m0");
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(at + TILE + i * 8192), "v"(v_at[i]), "s"(vrsrc), "s"(vo) : "memory", "m0");
    };
    request(0, 0);

    // ref: the row's reference (base-2 domain, the same in the four lanes of a row); sum: of this lane's keys
    float ref[2] = {-INFINITY, -INFINITY}, sum[2] = {0.0f, 0.0f};
    f32x4_acc o[2][FB];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int f = 0; f < FB; ++f) o[i][f] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};
    const int key = 4 * g + (r >> 2), flip = value_flip<D>(key);
    uint32_t v_read[FB];
#pragma unroll
    for (int f = 0; f < FB; ++f)
        v_read[f] = lds + TILE + (kg * KW + key) * ROW + (uint32_t)((((r & 3) * FB + f) >> 1) ^ flip) * 16 + (f & 1) * 8;

    auto tile_step = [&](int tile, int stage, auto edge_c) __attribute__((always_inline)) {
        constexpr bool EDGE = decltype(edge_c)::value;  // keys past the last one, or beyond some row's diagonal
        const unsigned char *kt = tiles + stage * STAGE;
        f32x4_acc s[2][NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            vec8 kf[KS];
#pragma unroll
            for (int k = 0; k < KS; ++k) kf[k] = *reinterpret_cast<const vec8 *>(kt + swz_offset<ROW>(kg * KW + 16 * n + r, 4 * k + g));
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                s[i][n] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < KS; ++k) s[i][n] = mfma16(kf[k], qf[i][k], s[i][n]);
            }
            if (n % 2 == 1) __builtin_amdgcn_sched_barrier(0);  // (no more fragments in flight than two blocks' worth: registers)
        }
        if (EDGE) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int limit = min(N - 1, m0 + 16 * i + r + p.causal_off);
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        s[i][n][e] = tile * BN + kg * KW + 16 * n + 4 * g + e > limit ? -INFINITY : s[i][n][e];
            }
        }
        float top[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            top[i] = -INFINITY;
#pragma unroll
            for (int n = 0; n < NB; ++n) top[i] = fmaxf(fmaxf(fmaxf(top[i], s[i][n][0]), fmaxf(s[i][n][1], s[i][n][2])), s[i][n][3]);
            top[i] *= p.scale_log2;
        }
        if (__any(top[0] > ref[0] + kRescaleThreshold || top[1] > ref[1] + kRescaleThreshold)) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float now = fmaxf(ref[i], quarters_max(top[i]));
                const float by = ref[i] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ref[i] - now);
                ref[i] = now;
                sum[i] *= by;
#pragma unroll
                for (int f = 0; f < FB; ++f) o[i][f] *= by;
            }
        }
        vec8 pf[2][NB / 2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float minus = ref[i] == -INFINITY ? 0.0f : -ref[i];  // (a row that has seen no key yet: its scores are -inf)
#pragma unroll
            for (int t = 0; t < NB / 2; ++t) {
                float e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    e[j] = __builtin_amdgcn_exp2f(fmaf(s[i][2 * t + (j >> 2)][j & 3], p.scale_log2, minus));
                    sum[i] += e[j];
                }
                const u32x4 packed = {pack2<T>(e[0], e[1]), pack2<T>(e[2], e[3]), pack2<T>(e[4], e[5]), pack2<T>(e[6], e[7])};
                pf[i][t] = __builtin_bit_cast(vec8, packed);
            }
        }
        // values, four feature blocks at a time: lane i of a 16-lane group hands in 4 features of key i / 4 and receives 4 keys of one feature
        constexpr int VB = 4;
#pragma unroll
        for (int t = 0; t < NB / 2; ++t)
#pragma unroll
            for (int f0 = 0; f0 < FB; f0 += VB) {
                u32x2 lo[VB], hi[VB];
#pragma unroll
                for (int f = 0; f < VB; ++f) {
                    const uint32_t at = v_read[f0 + f] + stage * STAGE;
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo[f]) : "v"(at), "n"(t * 32 * ROW));
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi[f]) : "v"(at), "n"(t * 32 * ROW + 16 * ROW));
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int f = 0; f < VB; ++f) {
                    asm volatile("" : "+v"(lo[f]), "+v"(hi[f]));
                    const u32x4 v4 = {lo[f][0], lo[f][1], hi[f][0], hi[f][1]};
                    const vec8 vf = __builtin_bit_cast(vec8, v4);
                    o[0][f0 + f] = mfma16(vf, pf[0][t], o[0][f0 + f]);
                    o[1][f0 + f] = mfma16(vf, pf[1][t], o[1][f0 + f]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    for (int tile = 0; tile < n_tiles; ++tile) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();  // the tile has landed for everyone, and nobody reads the other stage any more
        if (tile + 1 < n_tiles) request(tile + 1, (tile + 1) & 1);
        const int first = tile * BN + kg * KW;
        if (first >= N || first > m0 + 31 + p.causal_off) continue;  // nothing for this wave's rows
        if (first + KW > N || first + KW - 1 > m0 + p.causal_off) tile_step(tile, tile & 1, BoolC<true>());
        else tile_step(tile, tile & 1, BoolC<false>());
    }

    // ---- the key groups meet: every wave leaves its accumulator in LDS (lane-major) and finishes FB / KG feature blocks of its rows
    __syncthreads();
    f32x4 *const mine = reinterpret_cast<f32x4 *>(tiles) + wave * (2 * FB * 64);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int f = 0; f < FB; ++f) mine[(i * FB + f) * 64 + lane] = f32x4{o[i][f][0], o[i][f][1], o[i][f][2], o[i][f][3]};
        const float total = quarters_sum(sum[i]);
        if (g == 0) {
            ref_of[wave][16 * i + r] = ref[i];
            sum_of[wave][16 * i + r] = total;
        }
    }
    __syncthreads();
    constexpr int SHARE = FB / KG, PART = SHARE > 1 ? 2 : 1;  // feature blocks of a wave, and of a store
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = m0 + 16 * i + r;
        if (m >= M) continue;
        float top = -INFINITY, total = 0.0f, by[KG];
#pragma unroll
        for (int w = 0; w < KG; ++w) top = fmaxf(top, ref_of[w * QG + qg][16 * i + r]);
#pragma unroll
        for (int w = 0; w < KG; ++w) {
            const float rw = ref_of[w * QG + qg][16 * i + r];
            by[w] = rw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(rw - top);
            total = fmaf(by[w], sum_of[w * QG + qg][16 * i + r], total);
        }
        const float inv = 1.0f / total;
        T *orow = static_cast<T *>(p.o) + b * p.os[0] + h * p.os[1] + (int64_t)m * p.os[2] + 4 * FB * g;
#pragma unroll
        for (int f0 = 0; f0 < SHARE; f0 += PART) {
            float y[4 * PART];
#pragma unroll
            for (int k = 0; k < PART; ++k) {
                const int f = kg * SHARE + f0 + k;
                f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int w = 0; w < KG; ++w) {
                    const f32x4 v = (reinterpret_cast<const f32x4 *>(tiles) + (w * QG + qg) * (2 * FB * 64))[(i * FB + f) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[e] = fmaf(by[w], v[e], a[e]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) y[4 * k + e] = a[e] * inv;
            }
            T *at = orow + 4 * (kg * SHARE + f0);
            if constexpr (PART == 2)
                *reinterpret_cast<u32x4 *>(at) = u32x4{pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3]), pack2<T>(y[4], y[5]), pack2<T>(y[6], y[7])};
            else *reinterpret_cast<u32x2 *>(at) = u32x2{pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])};
        }
    }
}

template <typename T, int D>
static void launch_split(AttnParams p, hipStream_t st) {
    constexpr int LDS = 2 * 2 * 128 * D * 2;
    p.nq_tiles = (p.M + 63) / 64;
    auto kern = attention_split_kernel<T, D>;
    static bool attr_done = false;  // benign race: the attribute call is idempotent
    if (!attr_done) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        attr_done = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.B * p.H * p.nq_tiles)), dim3(512), LDS, st, p);
}

void run_attention_split(const AttnParams &p, int D, int dtype, hipStream_t st) {
    if (dtype == KERNL_F16) D == 64 ? launch_split<f16, 64>(p, st) : launch_split<f16, 128>(p, st);
    else D == 64 ? launch_split<bf16, 64>(p, st) : launch_split<bf16, 128>(p, st);
}

}  // namespace kernl
