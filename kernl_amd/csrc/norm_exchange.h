// linear + residual + LayerNorm in ONE launch, for rows whose output columns are spread over several workgroups: the workgroups of a
// row tile exchange the statistics of their columns — 8 bytes a row and column tile — and each normalises the sums it still holds in
// registers.  What a launch of its own behind the product costs is the launch, the sums' way to memory and back, and their rounding
// to 16 bits on that way; the exchange is one store and one load of a few KB at agent scope.
//
// Words.  For every column tile a word a row: (mean, sum of squared deviations) of the row's columns in that tile, both fp32, the second
// with its sign bit set, so that no word that was written is zero.  In front of them one word a row tile for notes.  All are zero when a
// launch starts: the caller hands in two regions by turns, and a launch clears the one that the NEXT launch takes.  They are written and
// read with relaxed 8-byte accesses at agent scope, which the XCDs' L2 caches do not hold back.
//
// Every wait ends.  A workgroup looks for the words of the others `patience` times.  They all lie in the same round of the grid, so that
// in ordinary use they arrive within a microsecond or two; but nothing guarantees that they run at the same time (other streams,
// other processes).  A workgroup whose patience runs out stores its sums in fp32, notes that it leaves (bit t of the note word for
// column tile t), looks once more and, if words are still missing, ends.  A workgroup that has found all words reads the note word once
// its own words have arrived in memory, and normalises the tiles of those that left.  So either the leaving one's last look finds the
// words of the last to publish, or that one finds the note: it has every word, and never leaves.  (Both may happen, and several may
// find a note: the same values are written twice.)
#pragma once

#include "norm_fold.h"

namespace kernl {

constexpr int exchange_lanes(int bm, int threads) { return threads / bm >= 8 ? 8 : threads / bm >= 4 ? 4 : threads / bm >= 2 ? 2 : 1; }  // lanes that look for a row's words
constexpr int exchange_most(int lanes) { return lanes < 4 ? 4 * lanes : 32; }  // column tiles whose words they can hold
constexpr int kExchangePatience = 1 << 9;    // looks, at about a microsecond each

struct NormExchange : NormFold {             // residual, res_rs, gamma, beta and eps of the norm behind the product
    uint64_t *words = nullptr;               // this launch's region, zeros
    uint64_t *clear = nullptr;               // the region of the launch behind it
    int clear_words = 0;
    int patience = kExchangePatience;
    float *sums = nullptr;                   // [M, N]: rows of the workgroups that leave
    float inv_n = 1.0f;                      // 1 / N
};

// words of one region
static inline int64_t exchange_words(int64_t tiles_m, int64_t tiles_n, int64_t bm) { return tiles_m * (1 + tiles_n * bm); }

__device__ __forceinline__ void store_agent(uint64_t *p, uint64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint64_t load_agent(uint64_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// (A release fence would write back the whole L2: the words go past it, and have arrived when the store counter is zero.)
__device__ __forceinline__ void published_words_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// the region of the next launch; threads 0 .. threads - 1 of every workgroup of the grid take part
__device__ __forceinline__ void exchange_clear(const NormExchange &nx, int tid, int threads) {
    for (int i = (int)blockIdx.x * threads + tid; i < nx.clear_words; i += (int)gridDim.x * threads) nx.clear[i] = 0;
}

// The exchange of one workgroup of a row tile of BM rows, `tiles` column tiles of BN columns.  T neighbouring lanes look for the words of a row.
template <int BM, int BN, int T>
struct RowExchange {
    static_assert(T == 1 || T == 2 || T == 4 || T == 8, "lanes a row");
    static constexpr int PER = exchange_most(T) / T;  // up to 32 column tiles: a note bit each
    uint64_t *notes, *words;
    int tiles;
    __device__ __forceinline__ RowExchange(const NormExchange &nx, int tile_m, int tiles_m, int tiles_n)
        : notes(nx.words + tile_m), words(nx.words + tiles_m + (int64_t)tile_m * tiles_n * BM), tiles(tiles_n) {}

    __device__ __forceinline__ void publish(int tile_n, int row, float mean, float m2) const {
        const uint32_t hi = __builtin_bit_cast(uint32_t, m2) | 0x80000000u;
        store_agent(words + (int64_t)tile_n * BM + row, (uint64_t)hi << 32 | __builtin_bit_cast(uint32_t, mean));
    }
    // by one thread, once the workgroup's sums are in memory; what it reads behind it is read behind the note
    __device__ __forceinline__ void note_leaving(int tile_n) const {
        const uint64_t before = __hip_atomic_fetch_or(notes, (uint64_t)1 << tile_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" :: "v"((uint32_t)before) : "memory");  // (waited for)
    }
    // (mean, 1 / std) of the row, to each of its T lanes; false if a word of one of the wave's rows is not there after `patience` more looks
    __device__ __forceinline__ bool look(int row, int t, int patience, float inv_n, float eps, f32x2 &norm) const {
        uint64_t w[PER];
        for (;;) {
            bool there = true;
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                w[q] = 0;
                if (t + T * q < tiles) w[q] = load_agent(words + (int64_t)(t + T * q) * BM + row);
            }
#pragma unroll
            for (int q = 0; q < PER; ++q)
                if (t + T * q < tiles) there = there && w[q] != 0;
            if (__all(there)) break;
            if (patience-- <= 0) return false;
            __builtin_amdgcn_s_sleep(1);
        }
        auto lanes_sum = [](float v) __attribute__((always_inline)) {
            if (T >= 2) v += dpp_mov<0xB1>(v);
            if (T >= 4) v += dpp_mov<0x4E>(v);
            if (T >= 8) v += dpp_mov<0x141>(v);
            return v;
        };
        float mean = 0.0f, m2 = 0.0f;
#pragma unroll
        for (int q = 0; q < PER; ++q)
            if (t + T * q < tiles) mean += __builtin_bit_cast(float, (uint32_t)w[q]);
        mean = lanes_sum(mean) * ((float)BN * inv_n);
#pragma unroll
        for (int q = 0; q < PER; ++q)
            if (t + T * q < tiles) {
                const float d = __builtin_bit_cast(float, (uint32_t)w[q]) - mean;
                m2 += fmaf((float)BN * d, d, __builtin_bit_cast(float, (uint32_t)(w[q] >> 32) & 0x7FFFFFFFu));
            }
        norm = f32x2{mean, rsqrtf(fmaf(lanes_sum(m2), inv_n, eps))};
        return true;
    }
};

// one value of the result, in fp32: rounded to it before it is to 16 bits wherever it is computed (no mixed-precision product)
__device__ __forceinline__ float exchange_normalised(float v, f32x2 factors, float gamma, float beta) {
    float y = fmaf((v - factors[0]) * factors[1], gamma, beta);
    asm("" : "+v"(y));
    return y;
}

// the tiles that were left (bits of `left`), normalised from memory by `threads` threads
template <typename T, int BM, int BN>
__device__ __forceinline__ void exchange_finish_others(const NormExchange &nx, uint64_t left, const f32x2 *row_norm, T *out, int64_t out_rs, int m0,
                                                       int M, int N, int tid, int threads) {
    while (left != 0) {
        const int n0 = __builtin_ctzll(left) * BN;
        left &= left - 1;
#pragma unroll 1
        for (int at = tid; at < BM * (BN / 2); at += threads) {
            const int row = at / (BN / 2), m = m0 + row, n = n0 + at % (BN / 2) * 2;
            if (m >= M) continue;
            const uint64_t pair = load_agent(reinterpret_cast<uint64_t *>(nx.sums + (int64_t)m * N + n));
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float v = __builtin_bit_cast(float, (uint32_t)(pair >> (32 * e)));
                const float beta = nx.beta != nullptr ? to_float(static_cast<const T *>(nx.beta)[n + e]) : 0.0f;
                out[(int64_t)m * out_rs + n + e] = from_float<T>(exchange_normalised(v, row_norm[row], to_float(static_cast<const T *>(nx.gamma)[n + e]), beta));
            }
        }
    }
}

}  // namespace kernl
