// Tiles of the linear layer for middling problems: what a workgroup does with one (linear_mid.hip says why it looks like this).
#pragma once

#include "linear_kernels.h"
#include "norm_exchange.h"

namespace kernl {

// tile shape, grid of the multiplying waves (eight or four) and ring depth of one build
template <int BM_, int BN_, int WM_, int WN_, int S_>
struct MidTile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = S_;
    static constexpr int BK = 64, RB = BK * 2, LOADERS = 4, MULS = WM * WN, WAVES = MULS + LOADERS;
    static constexpr int TM = BM / WM, TN = BN / WN, NBM = TM / 16, NBN = TN / 16;
    static constexpr bool X_AHEAD = TM * TN < 96 * 48;  // registers for two sets of x fragments
    static constexpr bool SPREAD = MULS == 4 || TM * TN >= 64 * 64;  // fragment reads between the matrix instructions (see multiply)
    static constexpr bool STAGED = TM * TN >= 64 * 32;  // 16-bit results leave through LDS (see the epilogue)
    static constexpr int X_BYTES = BM * RB, STAGE = (BM + BN) * RB, LDS = S * STAGE;
    static constexpr int LX = BM / (8 * LOADERS), LW = BN / (8 * LOADERS), L = LX + LW;  // 1 KB loads of a loading wave per k-tile
    static_assert((MULS == 8 || MULS == 4) && LX * 8 * LOADERS == BM && LW * 8 * LOADERS == BN && LDS <= 160 * 1024 && (S == 3 || S == 4) && (S - 1) * L <= 63, "tile shape");
};

// How the tile grid is dealt to the 8 XCDs, each with an L2 of its own: as 2^xm_shift x 8 / 2^xm_shift blocks of per_m x per_n tiles,
// so that an XCD reads a part of x AND a part of the weight (1024 x 768 x 3072 in 64 x 64 tiles: 32 MB from the memory side instead of
// the 55 that a run of 24 tiles per XCD, which spans all of x, asks for).  per_m = 0: runs of tiles, the row tile fastest.
struct MidGrid {
    int xm_mask = 0, xm_shift = 0, per_m = 0, per_n = 0;
};

// which weight row of the tile LDS row `row` carries: the lane's blocks become consecutive output columns
template <bool GATED, int TN>
__device__ __forceinline__ int mid_weight_row(int row) {
    constexpr int NBN = TN / 16;
    const int wt = row / TN, rem = row % TN, j = rem / 16, rr = rem % 16;
    if (!GATED) return wt * TN + 4 * NBN * (rr >> 2) + 4 * j + (rr & 3);
    constexpr int H = NBN / 2;
    const int c = wt * (TN / 2) + 4 * H * (rr >> 2) + 4 * (j % (H > 0 ? H : 1)) + (rr & 3);
    return 64 * (c >> 5) + (c & 31) + 32 * (j / (H > 0 ? H : 1));
}

// The residual of a lane's rows and columns, four 16-bit values a block; requested in front of the main loop where there are registers for it
template <typename Cfg>
constexpr bool mid_residual_ahead() { return Cfg::NBM * Cfg::NBN <= 12; }
template <typename T, typename Cfg>
__device__ __forceinline__ void mid_residual(const NormExchange &norm, u32x2 (&res)[Cfg::NBM][Cfg::NBN], int m0, int n0, int M, int wave, int lane) {
    const int m = m0 + wave % Cfg::WM * Cfg::TM + (lane & 15), n = n0 + wave / Cfg::WM * Cfg::TN + 4 * Cfg::NBN * (lane >> 4);
#pragma unroll
    for (int i = 0; i < Cfg::NBM; ++i)
#pragma unroll
        for (int j = 0; j < Cfg::NBN; ++j)
            res[i][j] = *reinterpret_cast<const u32x2 *>(static_cast<const T *>(norm.residual) + (int64_t)min(m + 16 * i, M - 1) * norm.res_rs + n + 4 * j);
}

// The epilogue of a norm: sums + bias + residual, the rows' statistics, the exchange, and the normalised rows through LDS.  What bounds it is
// the exchange, a store and a load at agent scope (about 1.5 us); gamma and beta travel beside it.
template <typename T, typename Cfg>
__device__ __forceinline__ void linear_mid_norm_rows(const NormExchange &norm, f32x4_acc (&acc)[Cfg::NBM][Cfg::NBN], const u32x2 (&bias_raw)[Cfg::NBN],
                                                     u32x2 (&res)[Cfg::NBM][Cfg::NBN], unsigned char *smem, T *out, int64_t out_rs, int M, int N, int tiles_m, int tile_m,
                                                     int tile_n, int tid) {
    typedef typename Vec8<T>::type vec8;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, TM = Cfg::TM, TN = Cfg::TN, NBM = Cfg::NBM, NBN = Cfg::NBN, C = 4 * NBN, LANES = exchange_lanes(BM, Cfg::MULS * 64);
    constexpr int PITCH = TN * 2 + 16, CH = TN / 8, ITER = (TM * CH + 63) / 64;
    // LDS: the waves' results, the statistics of the waves' columns, the rows' factors, and what the workgroup has to agree on
    constexpr int STATS = Cfg::MULS * TM * PITCH, FACTORS = STATS + Cfg::WN * BM * 8, VERDICT = FACTORS + BM * 8;
    static_assert(VERDICT + 16 <= Cfg::LDS, "all of it in the ring");
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wave_m = wave % Cfg::WM, wave_n = wave / Cfg::WM, r = lane & 15, g = lane >> 4;
    const int m0 = tile_m * BM, mw = m0 + wave_m * TM, nl = tile_n * BN + wave_n * TN + C * g;  // the wave's first row, the lane's first column
    f32x2 *const wave_stats = reinterpret_cast<f32x2 *>(smem + STATS), *const row_norm = reinterpret_cast<f32x2 *>(smem + FACTORS);
    uint32_t *const failed = reinterpret_cast<uint32_t *>(smem + VERDICT);
    const RowExchange<BM, BN, LANES> exchange(norm, tile_m, tiles_m, N / BN);
    if (!mid_residual_ahead<Cfg>()) mid_residual<T, Cfg>(norm, res, m0, tile_n * BN, M, wave, lane);
    if (tid == 0) *failed = 0;
#pragma unroll
    for (int i = 0; i < NBM; ++i) {
        float sum = 0.0f, m2 = 0.0f;
#pragma unroll
        for (int j = 0; j < NBN; ++j) {
            float b[4], h[4];
            unpack4<T>(bias_raw[j], b);
            unpack4<T>(res[i][j], h);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[i][j][e] = acc[i][j][e] + b[e] + h[e];
                sum += acc[i][j][e];
            }
        }
        const float mean = rows4_sum(sum) * (1.0f / TN);
#pragma unroll
        for (int j = 0; j < NBN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) m2 = fmaf(acc[i][j][e] - mean, acc[i][j][e] - mean, m2);
        m2 = rows4_sum(m2);
        if (g == 0) wave_stats[wave_n * BM + wave_m * TM + 16 * i + r] = f32x2{mean, m2};
    }
    u32x2 gam[NBN], bet[NBN];
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
        gam[j] = *reinterpret_cast<const u32x2 *>(static_cast<const T *>(norm.gamma) + nl + 4 * j);
        bet[j] = norm.beta != nullptr ? *reinterpret_cast<const u32x2 *>(static_cast<const T *>(norm.beta) + nl + 4 * j) : u32x2{0, 0};
    }
    __syncthreads();
    if (tid < BM) {  // a thread a row, whole waves
        float mean = 0.0f, m2 = 0.0f;
        f32x2 part[Cfg::WN];
#pragma unroll
        for (int w = 0; w < Cfg::WN; ++w) {
            part[w] = wave_stats[w * BM + tid];
            mean += part[w][0];
        }
        mean *= 1.0f / Cfg::WN;
#pragma unroll
        for (int w = 0; w < Cfg::WN; ++w) m2 += fmaf((float)TN * (part[w][0] - mean), part[w][0] - mean, part[w][1]);
        exchange.publish(tile_n, tid, mean, m2);
    }
    // (mean, 1 / std) of the rows to LDS
    auto factors = [&](int patience) __attribute__((always_inline)) {
        const int row = tid / LANES;
        f32x2 norm_of_row;
        if (row >= BM) return true;
        if (!exchange.look(row, tid % LANES, patience, norm.inv_n, norm.eps, norm_of_row)) return false;
        if (tid % LANES == 0) row_norm[row] = norm_of_row;
        return true;
    };
    if (!factors(norm.patience) && lane == 0) *failed = 1;
    published_words_landed();
    __syncthreads();
    if (*failed != 0) {
        // out of patience: the sums to memory, a note, and a last look
#pragma unroll
        for (int i = 0; i < NBM; ++i)
#pragma unroll
            for (int j = 0; j < NBN; ++j)
                if (mw + 16 * i + r < M)
#pragma unroll
                    for (int e = 0; e < 4; e += 2)
                        store_agent(reinterpret_cast<uint64_t *>(norm.sums + (int64_t)(mw + 16 * i + r) * N + nl + 4 * j + e),
                                    (uint64_t)__builtin_bit_cast(uint32_t, (float)acc[i][j][e + 1]) << 32 | __builtin_bit_cast(uint32_t, (float)acc[i][j][e]));
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
    unsigned char *const mine = smem + wave * (TM * PITCH);
#pragma unroll
    for (int i = 0; i < NBM; ++i) {
        const f32x2 f = row_norm[wave_m * TM + 16 * i + r];
#pragma unroll
        for (int j = 0; j < NBN; ++j) {
            float y[4], ga[4], be[4];
            unpack4<T>(gam[j], ga);
            unpack4<T>(bet[j], be);
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = exchange_normalised(acc[i][j][e], f, ga[e], be[e]);
            *reinterpret_cast<u32x2 *>(mine + (16 * i + r) * PITCH + (C * g + 4 * j) * 2) = u32x2{pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])};
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int at = it * 64 + lane, row = at / CH, c = at % CH;
        if ((TM * CH % 64 != 0 && row >= TM) || mw + row >= M) continue;
        *reinterpret_cast<vec8 *>(out + (int64_t)(mw + row) * out_rs + tile_n * BN + wave_n * TN + 8 * c) = *reinterpret_cast<const vec8 *>(mine + row * PITCH + c * 16);
    }
    if (left != 0) exchange_finish_others<T, BM, BN>(norm, left, row_norm, out, out_rs, m0, M, N, lane, 64);
}

// One tile by one workgroup.  Norm: NormExchange where the rows are added to a residual and normalised (norm_exchange.h), else NoNorm.
struct NoNorm {};
template <typename T, typename Cfg, bool GATED, typename Norm>
__device__ __forceinline__ void linear_mid_tile(const T *__restrict__ X, const T *__restrict__ W, const T *__restrict__ bias, T *__restrict__ out,
                  T *__restrict__ act_in, const float *__restrict__ row_scale, const T *__restrict__ residual, int M, int N, int K,
                  int64_t ldx, int64_t out_rs, int64_t out_cs, int64_t ai_rs, int64_t ai_cs, int64_t res_rs, int64_t res_cs, int act,
                  int tiles_m, const MidGrid &grid, float *__restrict__ part, int64_t part_rs, int range_kt, const Norm &norm) {
    constexpr bool NORM = std::is_same<Norm, NormExchange>::value;
    static_assert(!(NORM && GATED), "a norm follows a plain product");
    typedef typename Vec8<T>::type vec8;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, S = Cfg::S, NBM = Cfg::NBM, NBN = Cfg::NBN, STAGE = Cfg::STAGE, L = Cfg::L;
    constexpr int LX = Cfg::LX, LW = Cfg::LW, BK = Cfg::BK;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave % Cfg::WM, wave_n = wave / Cfg::WM;
    const int loader = wave % Cfg::LOADERS;
    const int r = lane & 15, g = lane >> 4;
    if constexpr (NORM)
        if (wave < Cfg::MULS) exchange_clear(norm, tid, Cfg::MULS * 64);
    // workgroup b runs on XCD b % 8, which works on a block of the tile grid of its own (or on a contiguous run of tiles)
    int tile_m, tile_n;
    if (grid.per_m != 0) {
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
        tile_m = (xcd & grid.xm_mask) * grid.per_m + slot % grid.per_m;
        tile_n = (xcd >> grid.xm_shift) * grid.per_n + slot / grid.per_m;
        if (tile_m >= tiles_m || tile_n * BN >= N) return;
    } else {
        const int tile = xcd_contiguous_index((int)blockIdx.x, (int)gridDim.x);
        tile_m = tile % tiles_m;
        tile_n = tile / tiles_m;
    }
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    // K split (part given): this workgroup's range of range_kt k-tiles
    const int64_t ldw = K;
    if (part != nullptr) {
        const int k_begin = (int)blockIdx.y * range_kt * BK;
        X += k_begin;
        W += k_begin;
        K = min(range_kt * BK, K - k_begin);
        part += (int64_t)blockIdx.y * M * part_rs;
    }
    // the order of the k-tiles, as in the wide kernels (linear_kernels.h) but for any K: whole groups of four are dealt
    const int turn = (tile_m + tile_n) & 3, k_dealt = K / (4 * BK) * 4;

    constexpr uint32_t kOutOfRange = 0x80000000u;
    const int rows_x = min(BM, M - m0), rows_w = min(BN, N - n0);
    const uint64_t xaddr = (uint64_t)(uintptr_t)(X + (int64_t)m0 * ldx);
    const uint64_t waddr = (uint64_t)(uintptr_t)(W + (int64_t)n0 * ldw);
    const u32x4 xrsrc = {(uint32_t)xaddr, (uint32_t)(xaddr >> 32) & 0xFFFFu, (uint32_t)((((int64_t)rows_x - 1) * ldx + K) * 2), 0x00020000u};
    const u32x4 wrsrc = {(uint32_t)waddr, (uint32_t)(waddr >> 32) & 0xFFFFu, (uint32_t)((((int64_t)rows_w - 1) * ldw + K) * 2), 0x00020000u};
    const int nk = (K + BK - 1) / BK, k_last = K - (nk - 1) * BK;
    // load i of a loading wave fills the 1 KB (8 rows) piece i * LOADERS + loader of the operand tile
    uint32_t xd[LX], wd[LW], tail_bits = 0;
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int q = (i * Cfg::LOADERS + loader) * 64 + lane, row = SmallTileMap::load_row(q), c = SmallTileMap::load_chunk(q);
        xd[i] = row < rows_x ? (uint32_t)(((int64_t)row * ldx + c * 8) * 2) : kOutOfRange;
        if (c * 8 < k_last) tail_bits |= 1u << i;
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int q = (i * Cfg::LOADERS + loader) * 64 + lane, row = mid_weight_row<GATED, Cfg::TN>(SmallTileMap::load_row(q)), c = SmallTileMap::load_chunk(q);
        wd[i] = row < rows_w ? (uint32_t)(((int64_t)row * ldw + c * 8) * 2) : kOutOfRange;
        if (c * 8 < k_last) tail_bits |= 1u << (LX + i);
    }
    typedef __attribute__((address_space(3))) void lds_void;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void *)smem + loader * 1024;
    auto load1 = [&](const u32x4 &rsrc, uint32_t off, uint32_t lds, int kbytes) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :: "s"(lds), "v"(off), "s"(rsrc), "s"(kbytes) : "memory", "m0");
    };
    auto clip = [&](uint32_t keep) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < LX; ++i) xd[i] = ((keep >> i) & 1u) != 0 ? xd[i] : kOutOfRange;
#pragma unroll
        for (int i = 0; i < LW; ++i) wd[i] = ((keep >> (LX + i)) & 1u) != 0 ? wd[i] : kOutOfRange;
    };
    auto request = [&](int kt, int stage) __attribute__((always_inline)) {
        if (kt == nk - 1) clip(tail_bits);
        const uint32_t base = lds_base + (uint32_t)stage * STAGE;
        const int kbytes = (kt < k_dealt ? kt ^ turn : kt) * BK * 2;
#pragma unroll
        for (int i = 0; i < LX; ++i) load1(xrsrc, xd[i], base + i * Cfg::LOADERS * 1024, kbytes);
#pragma unroll
        for (int i = 0; i < LW; ++i) load1(wrsrc, wd[i], base + Cfg::X_BYTES + i * Cfg::LOADERS * 1024, kbytes);
    };
    // (the blocks of a wave lie 16 rows apart, which leaves the swizzle as it is)
    int xoff[2], woff[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        xoff[st] = SmallTileMap::frag_offset(wave_m * Cfg::TM + r, st, g);
        woff[st] = Cfg::X_BYTES + SmallTileMap::frag_offset(wave_n * Cfg::TN + r, st, g);
    }
    f32x4_acc acc[NBM][NBN];
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) acc[i][j] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};

    // what the epilogue needs of the lane's rows and columns, requested before anything else: where it is used it would cost
    // a memory round trip
    constexpr int C = GATED ? 2 * NBN : 4 * NBN;  // consecutive output columns of a lane
    constexpr int V = C % 8 == 0 ? 8 : 4;         // columns per access
    typedef uint32_t words __attribute__((ext_vector_type(V / 2)));
    const int out_n = GATED ? N / 2 : N;
    u32x2 bias_raw[NBN];  // 16-bit values until the epilogue: registers are short in the large tiles
    const bool bias_vec = ((uintptr_t)bias & 7) == 0;
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
        const int n = n0 + mid_weight_row<GATED, Cfg::TN>(wave_n * Cfg::TN + 16 * j + 4 * g);
        if (bias != nullptr && bias_vec && n + 4 <= N) {
            bias_raw[j] = *reinterpret_cast<const u32x2 *>(bias + n);
            continue;
        }
        uint32_t b16[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) b16[e] = bias != nullptr && n + e < N ? reinterpret_cast<const uint16_t *>(bias)[n + e] : 0;
        bias_raw[j] = u32x2{b16[0] | b16[1] << 16, b16[2] | b16[3] << 16};
    }
    u32x2 res_raw[NORM ? NBM : 1][NORM ? NBN : 1];
    if constexpr (NORM && mid_residual_ahead<Cfg>()) {
        if (wave < Cfg::MULS) mid_residual<T, Cfg>(norm, res_raw, m0, n0, M, wave, lane);
    }
    auto wait_loads = [&](auto n_c) __attribute__((always_inline)) {
        constexpr int n = decltype(n_c)::value;
        __builtin_amdgcn_s_waitcnt(0x0F70 | (n & 15) | ((n >> 4) << 14));
    };
    if (wave >= Cfg::MULS) {
        // a loading wave: its stalls on the load path hold up neither the LDS reads nor the matrix instructions of the others.  Nothing
        // is requested beyond the last k-tile, so that after its barrier LDS is free for the epilogue without another one.
        auto landed = [&](int kt) __attribute__((always_inline)) {  // k-tile kt; at most S - 1 have been requested behind it
            const int behind = min(kt + S, nk) - 1 - kt;
            if (behind >= S - 1) wait_loads(IntC<(S - 1) * L>());
            else if (behind == S - 2) wait_loads(IntC<(S - 2) * L>());
            else if (S > 3 && behind == S - 3) wait_loads(IntC<(S - 3) * L>());
            else wait_loads(IntC<0>());
        };
#pragma unroll
        for (int kt = 0; kt < S; ++kt)
            if (kt < nk) request(kt, kt);
        landed(0);
        __syncthreads();
        int stage = 0;
        for (int kt = 0; kt < nk; ++kt) {
            // (before this iteration's request: one k-tile fewer behind the next one)
            if (kt + S < nk) wait_loads(IntC<(S - 2) * L>());
            else if (kt + 1 < nk) landed(kt + 1);
            __syncthreads();  // as below
            if (kt + S < nk) request(kt + S, stage);
            stage = stage == S - 1 ? 0 : stage + 1;
        }
        return;
    }

    // Fragments are read one k-step ahead, across the barrier.  The large tiles have no registers for a second set of x fragments: theirs
    // are overwritten one by one, each as soon as its row of blocks is done.
    constexpr int XB = Cfg::X_AHEAD ? 2 : 1;
    vec8 xf[XB][NBM], wf[2][NBN];
    auto read_x = [&](int st, const unsigned char *sb, int i) __attribute__((always_inline)) { xf[st % XB][i] = *reinterpret_cast<const vec8 *>(sb + xoff[st] + i * 2048); };
    auto read_w = [&](int st, const unsigned char *sb, int j) __attribute__((always_inline)) { wf[st][j] = *reinterpret_cast<const vec8 *>(sb + woff[st] + j * 2048); };
    // k-step st, and the fragments of the next one (of `stage`).  With eight waves and registers for both sets the reads go first: while one wave of a
    // SIMD requests, the other multiplies.  A SIMD's only multiplying wave, and waves of many blocks, request one behind every matrix
    // instruction, and x fragments that wait for registers behind the last one that needs the old: 128 x 256 and 256 x 128 tiles of
    // 4096 x 768 x 3072 34.8 -> 32.8 and 34.5 -> 32.0 us, of 1024 x 4096 x 4096 44.0 -> 41.8 and 44.2 -> 42.2.  (All others this way: 192 x 96 tiles of
    // 2048 x 768 x 3072 22.2 -> 22.8, 128 x 128 the same.)
    auto multiply = [&](int st, int stage) __attribute__((always_inline)) {
        const unsigned char *sb = smem + stage * STAGE;
        constexpr int READS = NBN + (XB == 2 ? NBM : 0), EACH = Cfg::SPREAD ? (READS + NBM * NBN - 1) / (NBM * NBN) : READS;
        auto read = [&](int q) __attribute__((always_inline)) {
            if (q < NBN) read_w(1 - st, sb, q);
            else read_x(1 - st, sb, q - NBN);
        };
        if (!Cfg::SPREAD) {
#pragma unroll
            for (int q = 0; q < READS; ++q) read(q);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < NBM * NBN; ++m) {
            const int i = m / NBN, j = m % NBN;
            acc[i][j] = mfma16(wf[st][j], xf[st % XB][i], acc[i][j]);
            if (!Cfg::SPREAD) continue;
#pragma unroll
            for (int q = m * EACH; q < (m + 1) * EACH && q < READS; ++q) read(q);
            if (XB == 1 && j == NBN - 1) read_x(1 - st, sb, i);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NBM; ++i) read_x(0, smem, i);
#pragma unroll
    for (int j = 0; j < NBN; ++j) read_w(0, smem, j);
    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
        const int next = stage == S - 1 ? 0 : stage + 1;
        multiply(0, stage);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __syncthreads();  // k-tile kt + 1 has landed for everyone, and nobody reads k-tile kt any more
        multiply(1, next);
        stage = next;
    }
    // (past the last barrier nothing lands in LDS any more and nobody reads a fragment that counts)

    // ---- epilogue.  A lane holds 4 to 24 consecutive columns of one row: stored from there, every 8 or 16 bytes are an access to a line
    // of their own, one a clock.  So a wave's results go through LDS (a region of its own, rows 16 bytes further apart than they are long)
    // and leave as whole rows of its block: the fp32 sums of a range of K always (333 x 4096 x 11008 in 192 x 128 tiles and four ranges,
    // 48 -> 44 us; 333 x 4096 x 4096 in 128 x 128 and two 22.8 -> 21.7), 16-bit results of the larger tiles (384 x 19200 x 64 in 192 x 192
    // 11.9 -> 9.7 us, 384 x 9600 x 64 in 192 x 96 8.1 -> 7.3, 333 x 32000 x 4096 in 192 x 128 101 -> 99).  The two smallest gain nothing
    // and would wait for LDS (231 x 2304 x 768 in 64 x 64 6.1 -> 6.2); they stage only what no vector store takes.
    constexpr int TNO = GATED ? Cfg::TN / 2 : Cfg::TN;  // output columns of a wave
    auto settle = [&]() __attribute__((always_inline)) {  // the wave's own LDS accesses, in order for the compiler too
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    };
    const int mw = m0 + wave_m * Cfg::TM;
    if (part != nullptr) {  // fp32 sums of the range, row-major; columns N .. part_rs - 1 hold zeros (their weight rows do)
        constexpr int PITCH = Cfg::TN * 4 + 16, CH = Cfg::TN / 4;
        static_assert(Cfg::MULS * 16 * PITCH <= Cfg::LDS, "a row block of every wave");
        unsigned char *mine = smem + wave * (16 * PITCH);
        const int nw = n0 + wave_n * Cfg::TN;
#pragma unroll
        for (int i = 0; i < NBM; ++i) {
#pragma unroll
            for (int j = 0; j < NBN; ++j) *reinterpret_cast<f32x4_acc *>(mine + r * PITCH + (C * g + 4 * j) * 4) = acc[i][j];
            settle();
#pragma unroll
            for (int it = 0; it < 16 * CH / 64; ++it) {
                const int at = it * 64 + lane, row = at / CH, c = at % CH, m = mw + 16 * i + row, n = nw + 4 * c;
                const f32x4_acc v = *reinterpret_cast<const f32x4_acc *>(mine + row * PITCH + c * 16);
                if (m < M && n < part_rs) *reinterpret_cast<f32x4_acc *>(part + (int64_t)m * part_rs + n) = v;
            }
            settle();
        }
        return;
    }
    if constexpr (NORM) {
        linear_mid_norm_rows<T, Cfg>(norm, acc, bias_raw, res_raw, smem, out, out_rs, M, N, tiles_m, tile_m, tile_n, tid);
        return;
    }
    constexpr int PITCH = TNO * 2 + 16, CH = TNO / 8, ITER = (Cfg::TM * CH + 63) / 64;
    static_assert(Cfg::MULS * Cfg::TM * PITCH <= Cfg::LDS, "the results of every wave");
    unsigned char *const mine = smem + wave * (Cfg::TM * PITCH);
    const int nw = (GATED ? n0 / 2 : n0) + wave_n * TNO;
    if (mw >= M || nw >= out_n) return;
    // the staged results to dst, + res rounded a second time as the sum of two 16-bit tensors is
    auto emit = [&](T *dst, int64_t rs, int64_t cs, const T *res) __attribute__((always_inline)) {
        settle();
        const bool rows16 = cs == 1 && (rs & 7) == 0 && ((uintptr_t)dst & 15) == 0 &&
                            (res == nullptr || (res_cs == 1 && (res_rs & 7) == 0 && ((uintptr_t)res & 15) == 0));
        if (rows16 && (nw + TNO <= out_n || (out_n & 7) == 0)) {
            vec8 rv[ITER];
            if (res != nullptr) {
#pragma unroll
                for (int it = 0; it < ITER; ++it) {
                    const int at = it * 64 + lane, row = at / CH, c = at % CH;
                    rv[it] = *reinterpret_cast<const vec8 *>(res + (int64_t)min(mw + row, M - 1) * res_rs + min(nw + 8 * c, out_n - 8));
                }
            }
#pragma unroll
            for (int it = 0; it < ITER; ++it) {
                const int at = it * 64 + lane, row = at / CH, c = at % CH;
                if ((Cfg::TM * CH % 64 != 0 && row >= Cfg::TM) || mw + row >= M || nw + 8 * c >= out_n) continue;
                vec8 v = *reinterpret_cast<const vec8 *>(mine + row * PITCH + c * 16);
                if (res != nullptr)
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = from_float<T>(to_float(v[e]) + to_float(rv[it][e]));
                *reinterpret_cast<vec8 *>(dst + (int64_t)(mw + row) * rs + nw + 8 * c) = v;
            }
        } else {
#pragma unroll 1
            for (int at = lane; at < Cfg::TM * TNO; at += 64) {
                const int row = at / TNO, c = at % TNO, m = mw + row, n = nw + c;
                if (m >= M || n >= out_n) continue;
                T v = *reinterpret_cast<const T *>(mine + row * PITCH + c * 2);
                if (res != nullptr) v = from_float<T>(to_float(v) + to_float(res[(int64_t)m * res_rs + (int64_t)n * res_cs]));
                dst[(int64_t)m * rs + (int64_t)n * cs] = v;
            }
        }
        settle();
    };
    float bz[NBN][4], scale[NBM];
#pragma unroll
    for (int j = 0; j < NBN; ++j) unpack4<T>(bias_raw[j], bz[j]);
#pragma unroll
    for (int i = 0; i < NBM; ++i) scale[i] = row_scale != nullptr ? row_scale[min(mw + 16 * i + r, M - 1)] : 1.0f;
    auto results = [&](auto act_c, int i, float (&y)[C]) __attribute__((always_inline)) {  // of the lane's row of row block i
        constexpr int ACT = decltype(act_c)::value;
#pragma unroll
        for (int j = 0; j < (GATED ? NBN / 2 : NBN); ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[4 * j + e] = apply_act16(fmaf(acc[i][j][e], scale[i], bz[j][e]), ACT);
                if (GATED) {
                    constexpr int H = GATED ? NBN / 2 : 0;
                    y[4 * j + e] *= fmaf(acc[i][(j + H) % NBN][e], scale[i], bz[(j + H) % NBN][e]);
                }
                asm("" : "+v"(y[4 * j + e]));  // rounded to fp32 before it is to T, in every form alike: no mixed-precision product
            }
    };
    auto packed = [&](const float *y) __attribute__((always_inline)) -> words {
        words w;
#pragma unroll
        for (int e = 0; e < V / 2; ++e) w[e] = pack2<T>(y[2 * e], y[2 * e + 1]);
        return w;
    };
    auto stage_as = [&](auto act_c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NBM; ++i) {
            float y[C];
            results(act_c, i, y);
#pragma unroll
            for (int c = 0; c < C; c += V) *reinterpret_cast<words *>(mine + (16 * i + r) * PITCH + (C * g + c) * 2) = packed(y + c);
        }
    };
    auto with_act = [&](auto then) __attribute__((always_inline)) {
        switch (act) {
            case KERNL_ACT_RELU: then(IntC<KERNL_ACT_RELU>()); break;
            case KERNL_ACT_TANH: then(IntC<KERNL_ACT_TANH>()); break;
            case KERNL_ACT_GELU_ERF: then(IntC<KERNL_ACT_GELU_ERF>()); break;
            case KERNL_ACT_GELU_TANH: then(IntC<KERNL_ACT_GELU_TANH>()); break;
            case KERNL_ACT_SILU: then(IntC<KERNL_ACT_SILU>()); break;
            default: then(IntC<KERNL_ACT_NONE>()); break;
        }
    };
    if constexpr (!Cfg::STAGED) {
        auto whole = [&](const void *p, int64_t rs, int64_t cs) __attribute__((always_inline)) { return p == nullptr || (cs == 1 && (rs & (V - 1)) == 0 && ((uintptr_t)p & (2 * V - 1)) == 0); };
        if (nw + TNO <= out_n && whole(out, out_rs, out_cs) && whole(act_in, ai_rs, ai_cs) && whole(residual, res_rs, res_cs)) {
            with_act([&](auto act_c) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NBM; ++i) {
                    const int m = mw + 16 * i + r;
                    if (m >= M) continue;
                    const int64_t n = nw + C * g;
                    float y[C];
                    if (!GATED && act_in != nullptr) {
                        results(IntC<KERNL_ACT_NONE>(), i, y);
#pragma unroll
                        for (int c = 0; c < C; c += V) *reinterpret_cast<words *>(act_in + m * ai_rs + n + c) = packed(y + c);
                    }
                    results(act_c, i, y);
                    if (residual != nullptr)
#pragma unroll
                        for (int c = 0; c < C; c += V) {
                            T rv[V];
                            *reinterpret_cast<words *>(rv) = *reinterpret_cast<const words *>(residual + m * res_rs + n + c);
#pragma unroll
                            for (int e = 0; e < V; ++e) y[c + e] = to_float(from_float<T>(y[c + e])) + to_float(rv[e]);
                        }
#pragma unroll
                    for (int c = 0; c < C; c += V) *reinterpret_cast<words *>(out + m * out_rs + n + c) = packed(y + c);
                }
            });
            return;
        }
    }
    if (!GATED && act_in != nullptr) {
        stage_as(IntC<KERNL_ACT_NONE>());
        emit(act_in, ai_rs, ai_cs, nullptr);
    }
    with_act(stage_as);
    emit(out, out_rs, out_cs, residual);
}

// the XCD blocks: as square in bytes as 8 blocks can be, where they take no more rounds than the tiles themselves; workgroups of the grid
template <typename Cfg>
static int mid_grid(int tiles_m, int tiles_n, int splits, MidGrid &grid) {
    int blocks = tiles_m * tiles_n;
    const int64_t all = (int64_t)blocks * splits;
    int64_t least = INT64_MAX;
    for (int s = 0; s <= 3; ++s) {
        const int xm = 1 << s, xn = 8 >> s, pm = (tiles_m + xm - 1) / xm, pn = (tiles_n + xn - 1) / xn;
        const int64_t bytes = (int64_t)pm * Cfg::BM + (int64_t)pn * Cfg::BN;
        if ((int64_t)pm * pn * splits > (all + 255) / 256 * 32 || bytes >= least) continue;
        least = bytes;
        grid.xm_mask = xm - 1; grid.xm_shift = s; grid.per_m = pm; grid.per_n = pn;
        blocks = 8 * pm * pn;
    }
    return blocks;
}

// the tiles, by the kernl_linear_force_tile value that forces them (and mid_tile_of names)
typedef MidTile<64, 64, 2, 2, 4> Mid64x64;      // 11   64 KB: two workgroups per CU
typedef MidTile<128, 64, 4, 2, 3> Mid128x64;    // 15   72 KB: two workgroups per CU
typedef MidTile<128, 128, 2, 4, 4> Mid128x128;  // 17
typedef MidTile<192, 128, 4, 2, 4> Mid192x128;  // 18
typedef MidTile<192, 192, 2, 4, 3> Mid192x192;  // 19   (six column blocks a wave spill without the gates' pairing,
typedef MidTile<192, 192, 4, 2, 3> Mid192x192g; //       which needs them even in number)
typedef MidTile<128, 256, 2, 4, 3> Mid128x256;  // 20
typedef MidTile<256, 128, 4, 2, 3> Mid256x128;  // 21
typedef MidTile<192, 96, 4, 2, 4> Mid192x96;    // 22   no gates: an odd number of column blocks

}  // namespace kernl
