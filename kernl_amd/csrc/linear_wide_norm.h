// What the 256-row wide kernel (linear_kernels.h) does with its sums where the rows are added to a residual and normalised (norm_exchange.h).
// A wave holds 128 rows x 16 NBN columns, four rows of a 16-row block and NBN consecutive columns a lane.  LDS: its last 8 KB, beside the
// stages (tile loads that were switched off still write zeros there).
#pragma once

#include "linear_kernels.h"
#include "norm_exchange.h"

namespace kernl {

constexpr int kWideStages = 2 * (256 + 256) * 128;       // bytes of the kernel's two stages
constexpr int kWideNormLds = kWideStages + 2 * 256 * 8 + 256 * 8 + 16;  // statistics of the waves' columns, the rows' factors, a verdict

template <typename F>
__device__ __forceinline__ void wide_blocks(F f) {  // (one call a block: the accumulators are only ever indexed by constants)
    f(IntC<0>()); f(IntC<1>()); f(IntC<2>()); f(IntC<3>());
    f(IntC<4>()); f(IntC<5>()); f(IntC<6>()); f(IntC<7>());
}

// What bounds it: 98 KB (NBN = 6) of residual and results a workgroup, the exchange (about 1.5 us) and some 25 vector instructions a value.
template <typename T, int NBN>
__device__ __forceinline__ void wide_norm_rows(const NormExchange &norm, f32x4_acc (&acc)[8][NBN], const float (&bf)[NBN], unsigned char *lds,
                                               T *__restrict__ out, int64_t out_rs, int M, int N, int tiles_m, int m0, int n0, int tid) {
    constexpr int BM = 256, BN = 32 * NBN, AHEAD = 3;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wave_m = wave & 1, wave_n = wave >> 1, l16 = lane & 15, g = lane >> 4;
    const int tile_n = n0 / BN, row0 = wave_m * 128 + 4 * g, n = n0 + wave_n * (NBN * 16) + l16 * NBN;  // the lane's first row of the tile, first column
    f32x2 *const wave_stats = reinterpret_cast<f32x2 *>(lds), *const row_norm = wave_stats + 2 * BM;
    uint32_t *const failed = reinterpret_cast<uint32_t *>(row_norm + BM);
    const RowExchange<BM, BN, 1> exchange(norm, m0 / BM, tiles_m, N / BN);
    typedef uint32_t words __attribute__((ext_vector_type(2)));
    static_assert(NBN == 8 || NBN == 6, "256 or 192 columns");
    auto row_words = [&](const void *base, int64_t at, uint32_t (&raw)[NBN / 2]) __attribute__((always_inline)) {
        const T *p = static_cast<const T *>(base) + at;
        if constexpr (NBN == 8) {
            const words a = *reinterpret_cast<const words *>(p), b = *reinterpret_cast<const words *>(p + 4);
            raw[0] = a[0], raw[1] = a[1], raw[2] = b[0], raw[3] = b[1];
        } else {
            const u32x3 a = *reinterpret_cast<const u32x3 *>(p);
            raw[0] = a[0], raw[1] = a[1], raw[2] = a[2];
        }
    };
    auto value = [](const uint32_t (&raw)[NBN / 2], int c) __attribute__((always_inline)) {
        return to_float(__builtin_bit_cast(T, (uint16_t)(raw[c >> 1] >> (16 * (c & 1)))));
    };
    uint32_t res[AHEAD][4][NBN / 2];  // of a ring of blocks
    auto fetch = [&](auto i_c) __attribute__((always_inline)) {
        constexpr int I = decltype(i_c)::value;
        if constexpr (I < 8)
#pragma unroll
            for (int v = 0; v < 4; ++v) row_words(norm.residual, (int64_t)min(m0 + row0 + 16 * I + v, M - 1) * norm.res_rs + n, res[I % AHEAD][v]);
    };
    if (tid == 0) *failed = 0;
    fetch(IntC<0>());
    fetch(IntC<1>());
    wide_blocks([&](auto i_c) __attribute__((always_inline)) {
        constexpr int I = decltype(i_c)::value;
        fetch(IntC<I + 2>());
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float sum = 0.0f, m2 = 0.0f;
#pragma unroll
            for (int c = 0; c < NBN; ++c) {
                acc[I][c][v] = acc[I][c][v] + bf[c] + value(res[I % AHEAD][v], c);
                sum += acc[I][c][v];
            }
            const float mean = row16_sum(sum) * (1.0f / (16 * NBN));
#pragma unroll
            for (int c = 0; c < NBN; ++c) m2 = fmaf(acc[I][c][v] - mean, acc[I][c][v] - mean, m2);
            m2 = row16_sum(m2);
            if (l16 == 0) wave_stats[wave_n * BM + row0 + 16 * I + v] = f32x2{mean, m2};
        }
    });
    uint32_t gam[NBN / 2], bet[NBN / 2] = {};
    row_words(norm.gamma, n, gam);
    if (norm.beta != nullptr) row_words(norm.beta, n, bet);
    __syncthreads();
    {  // a thread a row
        const f32x2 a = wave_stats[tid], b = wave_stats[BM + tid];
        const float mean = 0.5f * (a[0] + b[0]), da = a[0] - mean, db = b[0] - mean;
        exchange.publish(tile_n, tid, mean, a[1] + b[1] + (float)(16 * NBN) * fmaf(da, da, db * db));
    }
    // (mean, 1 / std) of the rows to LDS
    auto factors = [&](int patience) __attribute__((always_inline)) {
        f32x2 norm_of_row;
        if (!exchange.look(tid, 0, patience, norm.inv_n, norm.eps, norm_of_row)) return false;
        row_norm[tid] = norm_of_row;
        return true;
    };
    if (!factors(norm.patience) && lane == 0) *failed = 1;
    published_words_landed();
    __syncthreads();
    if (*failed != 0) {
        // out of patience: the sums to memory, a note, and a last look
        wide_blocks([&](auto i_c) __attribute__((always_inline)) {
            constexpr int I = decltype(i_c)::value;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + row0 + 16 * I + v;
                if (m < M)
#pragma unroll
                    for (int c = 0; c < NBN; c += 2)
                        store_agent(reinterpret_cast<uint64_t *>(norm.sums + (int64_t)m * N + n + c),
                                    (uint64_t)__builtin_bit_cast(uint32_t, (float)acc[I][c + 1][v]) << 32 | __builtin_bit_cast(uint32_t, (float)acc[I][c][v]));
            }
        });
        published_words_landed();
        __syncthreads();
        if (tid == 0) {
            exchange.note_leaving(tile_n);
            *failed = 0;
        }
        __syncthreads();
        if (!factors(0) && lane == 0) *failed = 1;
        __syncthreads();
        if (*failed != 0) return;
    }
    uint64_t left = 0;
    if (wave == 0) left = load_agent(exchange.notes);
    wide_blocks([&](auto i_c) __attribute__((always_inline)) {
        constexpr int I = decltype(i_c)::value;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = row0 + 16 * I + v;
            const f32x2 f = row_norm[row];
            float y[NBN];
#pragma unroll
            for (int c = 0; c < NBN; ++c) y[c] = exchange_normalised(acc[I][c][v], f, value(gam, c), value(bet, c));
            if (m0 + row < M) wide_store_row<T, NBN>(out + (int64_t)(m0 + row) * out_rs + n, y);
        }
    });
    if (left != 0) exchange_finish_others<T, BM, BN>(norm, left, row_norm, out, out_rs, m0, M, N, lane, 64);
}

}  // namespace kernl
