// Linear layer for SMALL problems: a few hundred rows against a weight of a few million elements (BERT-base at batch 1:
// 128 x 768 x 3072 and its siblings), where the big tile kernels have a handful of workgroups for 256 CUs and the
// split kernels pay for a second launch and for partial tiles larger than the output.
//
// Same operator as the other kernels (reference: `kernel_fma`, src/kernl/implementations/linear_layer.py:92-210 —
// C = act(A @ W^T + bias), optional store of the pre-activation); what differs is the shape of the work.  A workgroup of
// 4 waves (2 x 2) owns a 64 x 64 or 32 x 64 output tile over the WHOLE of K: one launch, no partial sums in memory,
// 50 to 256 workgroups.  Such a tile is 4 or 8 MFMAs per wave and 64-wide k-tile — the loop is bound by how fast the
// CU can pull its operand tiles (12 KB per k-tile) out of L2, i.e. by latency unless many k-tiles are in
// flight: operand tiles travel HBM/L2 -> LDS directly (buffer loads with the LDS flag, every lane fetching the 16-byte
// chunk that belongs at its LDS position under the XOR swizzle) through a ring of 8 stages, 7 k-tiles requested
// ahead, one barrier per k-tile and waits by count.  A last k-tile that reaches beyond K has the chunks that
// start there pointed out of range (zeros, in both operands).
#include "linear_kernels.h"
#include "norm_fold.h"

namespace kernl {

// Row statistics on their way to the epilogue: the pairs of a row tile lie in one piece of memory and travel to LDS in
// front of the first k-tile, `per_wave` KB-sized loads per wave (pieces past the end arrive as zeros or are not asked for).
constexpr int norm_stats_bytes(int bm) { return bm * 8 * (bm <= 32 ? 2 * kNormMaxGroups : kNormMaxGroups); }
template <int BM, int WAVES>
__device__ __forceinline__ void request_norm_stats(const NormFold &nf, int m0, int rows, uint32_t lds, int wave, int lane) {
    constexpr int PER_WAVE = norm_stats_bytes(BM) / 1024 / WAVES;
    static_assert(PER_WAVE >= 1, "whole KB per wave");
    const uint64_t addr = (uint64_t)(uintptr_t)(nf.in_stats + (int64_t)m0 * nf.in_groups * 2);
    const u32x4 rsrc = {(uint32_t)addr, (uint32_t)(addr >> 32) & 0xFFFFu, (uint32_t)(rows * nf.in_groups * 8), 0x00020000u};
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
        const int piece = wave * PER_WAVE + i;
        if (piece * 1024 < rows * nf.in_groups * 8)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :: "s"(lds + piece * 1024), "v"(piece * 1024 + lane * 16), "s"(rsrc) : "memory", "m0");
    }
}

constexpr int kSmallBK = 64;  // measured against 128-wide k-tiles in 6 / 4 stages: 5-10 % faster
// ring stages of the shared-tile kernel: 8 of them, or as many as fit 144 KB
constexpr int small_stages(int bm, int bn) { return (bm + bn) * kSmallBK * 2 * 8 <= 144 * 1024 ? 8 : (144 * 1024) / ((bm + bn) * kSmallBK * 2); }

template <typename T, int BM, int BN, int MODE>
__global__ void __launch_bounds__(256, 1)
linear_small_kernel(const T *__restrict__ X, const T *__restrict__ W, const T *__restrict__ bias, T *__restrict__ out,
                    T *__restrict__ act_in, int M, int N, int K, int64_t ldx, int64_t out_rs, int64_t out_cs,
                    int64_t ai_rs, int64_t ai_cs, int act, int tiles_m, NormFold nf) {
    typedef typename Vec8<T>::type vec8;
    constexpr int BK = kSmallBK, RB = BK * 2, CPR = BK / 8, S = small_stages(BM, BN), KSTEPS = BK / 32;
    static_assert(RB == SmallTileMap::ROW_BYTES && CPR == SmallTileMap::CHUNKS_PER_ROW, "tile rows as the tile map lays them out");
    constexpr int X_BYTES = BM * RB, W_BYTES = BN * RB, STAGE = X_BYTES + W_BYTES;
    constexpr int LX = BM * CPR / 256, LW = BN * CPR / 256, L = LX + LW;  // 1 KB loads per wave... per thread and stage
    constexpr int NBM = BM / 32, NBN = BN / 32;                            // 16 x 16 blocks per wave: rows of x, rows of w
    static_assert((BM == 32 || BM == 64) && (BN == 64 || BN == 128), "tile shapes");
    static_assert(S >= 3 && (S - 2) * L <= 63, "ring depth; the wait count must be encodable");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave & 1, wave_n = wave >> 1;
    const int r = lane & 15, g = lane >> 4;
    // tiles that share a weight tile (consecutive indices, the row tile running fastest) go to one XCD; with a single
    // row tile nothing is shared, and workgroups that run side by side had better read neighbouring weight rows
    const int tile = tiles_m > 1 ? xcd_contiguous_index((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;

    // ---- tile loads: load i of a wave fills the 1 KB of 16-byte chunks [(wave * loads + i) * 64, +64) of an operand
    // tile.  Rows beyond M / N are pointed out of the buffer's range and arrive as zeros.
    constexpr uint32_t kOutOfRange = 0x80000000u;
    const int rows_x = min(BM, M - m0), rows_w = min(BN, N - n0);
    const uint64_t xaddr = (uint64_t)(uintptr_t)(X + (int64_t)m0 * ldx);
    const uint64_t waddr = (uint64_t)(uintptr_t)(W + (int64_t)n0 * K);
    const u32x4 xrsrc = {(uint32_t)xaddr, (uint32_t)(xaddr >> 32) & 0xFFFFu,
                         (uint32_t)((((int64_t)rows_x - 1) * ldx + K) * 2), 0x00020000u};
    const u32x4 wrsrc = {(uint32_t)waddr, (uint32_t)(waddr >> 32) & 0xFFFFu, (uint32_t)((int64_t)rows_w * K * 2),
                         0x00020000u};
    uint32_t xd[LX], wd[LW];
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int q = (wave * LX + i) * 64 + lane;
        const int row = SmallTileMap::load_row(q), c = SmallTileMap::load_chunk(q);
        xd[i] = row < rows_x ? (uint32_t)(((int64_t)row * ldx + c * 8) * 2) : kOutOfRange;
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int q = (wave * LW + i) * 64 + lane;
        const int row = SmallTileMap::load_row(q), c = SmallTileMap::load_chunk(q);
        wd[i] = row < rows_w ? (uint32_t)(((int64_t)row * K + c * 8) * 2) : kOutOfRange;
    }
    // bit l of tail_bits: the chunk load l of this lane fetches starts below K in the last k-tile
    const int nk = (K + BK - 1) / BK;
    const int k_last = K - (nk - 1) * BK;
    uint32_t tail_bits = 0;
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int q = (wave * LX + i) * 64 + lane;
        if (SmallTileMap::load_chunk(q) * 8 < k_last) tail_bits |= 1u << i;
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int q = (wave * LW + i) * 64 + lane;
        if (SmallTileMap::load_chunk(q) * 8 < k_last) tail_bits |= 1u << (LX + i);
    }
    typedef __attribute__((address_space(3))) void lds_void;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void *)smem;
    // inline assembly on purpose: the compiler would make every later LDS read wait for loads it sees writing LDS
    auto load1 = [&](const u32x4 &rsrc, uint32_t off, uint32_t lds, int kbytes) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :: "s"(lds), "v"(off), "s"(rsrc), "s"(kbytes) : "memory", "m0");
    };
    // The offsets are clipped in place, under a branch taken twice per workgroup: to the chunks below K when the last
    // k-tile is requested, to nothing at the first request past it (the counts stay exact: every slot issues its loads).
    // A select per load would put three VALU instructions per load into every k-tile.
    auto clip = [&](uint32_t keep) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");  // keeps this a branch: without it the compiler turns the block into selects
#pragma unroll
        for (int i = 0; i < LX; ++i) xd[i] = ((keep >> i) & 1u) != 0 ? xd[i] : kOutOfRange;
#pragma unroll
        for (int i = 0; i < LW; ++i) wd[i] = ((keep >> (LX + i)) & 1u) != 0 ? wd[i] : kOutOfRange;
    };
    // k-tile kt into stage `stage`
    auto request = [&](int kt, int stage) __attribute__((always_inline)) {
        if (kt == nk - 1 || kt == nk) clip(kt == nk ? 0u : tail_bits);
        const uint32_t base = lds_base + (uint32_t)stage * STAGE;
        const int kbytes = kt < nk ? kt * BK * 2 : 0;
#pragma unroll
        for (int i = 0; i < LX; ++i) load1(xrsrc, xd[i], base + (wave * LX + i) * 1024, kbytes);
#pragma unroll
        for (int i = 0; i < LW; ++i) load1(wrsrc, wd[i], base + X_BYTES + (wave * LW + i) * 1024, kbytes);
    };

    // LDS byte offsets of this lane's fragments inside a stage: block rows, k-step st, 8 k-values per 16-byte unit
    int xoff[KSTEPS][NBM], woff[KSTEPS][NBN];
#pragma unroll
    for (int st = 0; st < KSTEPS; ++st) {
#pragma unroll
        for (int i = 0; i < NBM; ++i) xoff[st][i] = SmallTileMap::frag_offset(wave_m * (BM / 2) + 16 * i + r, st, g);
#pragma unroll
        for (int j = 0; j < NBN; ++j) woff[st][j] = X_BYTES + SmallTileMap::frag_offset(wave_n * (BN / 2) + 16 * j + r, st, g);
    }

    f32x4_acc acc[NBM][NBN];  // block (i, j): lane (r, g) holds x row 16 i + r, output columns 16 j + 4 g .. + 3
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) acc[i][j] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};
    // what the epilogue needs of the lane's rows and columns, requested before anything else: fetched where it is used,
    // every block of the epilogue would cost the wave a memory round trip of its own
    float bz[NBN][4];
    f32x4 cs[MODE == kNormApply ? NBN : 1];
    u32x2 res[MODE == kNormAdd ? NBM : 1][MODE == kNormAdd ? NBN : 1], gam[MODE == kNormAdd ? NBN : 1], bet[MODE == kNormAdd ? NBN : 1];
    const bool bias_vec = ((uintptr_t)bias & 7) == 0;
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
        const int n = n0 + wave_n * (BN / 2) + 16 * j + 4 * g;
        if (MODE == kNormApply) {
            const bool in = n < N;  // (N is a multiple of 32 with a norm)
            const f32x4 b32 = in ? *reinterpret_cast<const f32x4 *>(nf.bias32 + n) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            cs[j] = in ? *reinterpret_cast<const f32x4 *>(nf.colsum + n) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < 4; ++e) bz[j][e] = b32[e];
        } else {
            load_bias4<T>(bias, n, N, bias_vec, bz[j]);
        }
        if (MODE == kNormAdd) {
#pragma unroll
            for (int i = 0; i < NBM; ++i) {
                const int m = m0 + wave_m * (BM / 2) + 16 * i + r;
                res[i][j] = m < M && n < N ? *reinterpret_cast<const u32x2 *>(static_cast<const T *>(nf.residual) + (int64_t)m * nf.res_rs + n) : u32x2{0, 0};
            }
            if (nf.in_stats != nullptr) {
                gam[j] = n < N ? *reinterpret_cast<const u32x2 *>(static_cast<const T *>(nf.gamma) + n) : u32x2{0, 0};
                bet[j] = n < N && nf.beta != nullptr ? *reinterpret_cast<const u32x2 *>(static_cast<const T *>(nf.beta) + n) : u32x2{0, 0};
            }
        }
    }
    const bool row_stats = MODE == kNormApply || (MODE == kNormAdd && nf.in_stats != nullptr);
    if (MODE != kNormNone && row_stats) request_norm_stats<BM, 4>(nf, m0, rows_x, lds_base + S * STAGE, wave, lane);

#pragma unroll
    for (int kt = 0; kt < S - 1; ++kt) request(kt, kt);
    int stage = 0;  // stage of k-tile kt
    for (int kt = 0; kt < nk; ++kt) {
        // this wave's loads of k-tile kt have landed when at most (S - 2) stages' worth are still outstanding
        __builtin_amdgcn_s_waitcnt(0x0F70 | (((S - 2) * L) & 15) | ((((S - 2) * L) >> 4) << 14));
        __syncthreads();  // ... everyone's have, and nobody reads the stage of k-tile kt - 1 any more
        request(kt + S - 1, stage == 0 ? S - 1 : stage - 1);
        const unsigned char *sb = smem + stage * STAGE;
        // all fragment reads of the k-tile go out together; the MFMAs of a k-step wait for theirs only
        vec8 xf[KSTEPS][NBM], wf[KSTEPS][NBN];
#pragma unroll
        for (int st = 0; st < KSTEPS; ++st) {
#pragma unroll
            for (int i = 0; i < NBM; ++i) xf[st][i] = *reinterpret_cast<const vec8 *>(sb + xoff[st][i]);
#pragma unroll
            for (int j = 0; j < NBN; ++j) wf[st][j] = *reinterpret_cast<const vec8 *>(sb + woff[st][j]);
        }
#pragma unroll
        for (int st = 0; st < KSTEPS; ++st)
#pragma unroll
            for (int i = 0; i < NBM; ++i)
#pragma unroll
                for (int j = 0; j < NBN; ++j) acc[i][j] = mfma16(wf[st][j], xf[st][i], acc[i][j]);
        stage = stage == S - 1 ? 0 : stage + 1;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the out-of-range requests of the last rounds are done with before the LDS goes away

    if (MODE != kNormNone) {
        // mean and 1 / std of the lane's rows: the four lanes of a row take a quarter of its statistics pairs each
        float mean[NBM], rstd[NBM];
        if (row_stats) {
            const unsigned char *st = smem + S * STAGE;
            const int groups = nf.in_groups;
#pragma unroll
            for (int i = 0; i < NBM; ++i) {
                const f32x2 *row = reinterpret_cast<const f32x2 *>(st) + (wave_m * (BM / 2) + 16 * i + r) * groups;
                const float pivot = row[0][0] * nf.inv_group;
                NormMerge mg;
                f32x2 pairs[kNormMaxGroups / 2];  // (read together: one after the other each costs an LDS round trip)
#pragma unroll
                for (int q = 0; q < kNormMaxGroups / 2; ++q) pairs[q] = row[4 * q + g < groups ? 4 * q + g : 0];
#pragma unroll
                for (int q = 0; q < kNormMaxGroups / 2; ++q)
                    if (4 * q + g < groups) mg.take(pairs[q], pivot, nf.inv_group);
                mg.d = halves32_sum(mg.d + __shfl_xor(mg.d, 16));
                mg.dd = halves32_sum(mg.dd + __shfl_xor(mg.dd, 16));
                mg.m2 = halves32_sum(mg.m2 + __shfl_xor(mg.m2, 16));
                const f32x2 norm = mg.finish(pivot, nf);
                mean[i] = norm[0];
                rstd[i] = norm[1];
            }
        }
        auto finish_norm = [&](auto act_c) __attribute__((always_inline)) {
            constexpr int ACT = decltype(act_c)::value;
#pragma unroll
            for (int i = 0; i < NBM; ++i) {
                const int m = m0 + wave_m * (BM / 2) + 16 * i + r;
                float y[NBN][4];
#pragma unroll
                for (int j = 0; j < NBN; ++j) {
                    const int n = n0 + wave_n * (BN / 2) + 16 * j + 4 * g;
                    float h[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    if (MODE == kNormAdd) {
                        unpack4<T>(res[i][j], h);
                        if (row_stats) {
                            float gm[4], bt[4];
                            unpack4<T>(gam[j], gm);
                            unpack4<T>(bet[j], bt);
#pragma unroll
                            for (int e = 0; e < 4; ++e) h[e] = fmaf((h[e] - mean[i]) * rstd[i], gm[e], bt[e]);
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (MODE == kNormApply) y[j][e] = apply_act16(fmaf(fmaf(-mean[i], cs[j][e], acc[i][j][e]), rstd[i], bz[j][e]), ACT);
                        else y[j][e] = to_float(from_float<T>(acc[i][j][e] + bz[j][e] + h[e]));
                    }
                    if (m < M && n < N)
                        *reinterpret_cast<u32x2 *>(out + (int64_t)m * out_rs + n) = u32x2{pack2<T>(y[j][0], y[j][1]), pack2<T>(y[j][2], y[j][3])};
                }
                if (MODE == kNormAdd) {
                    // statistics of the stored values: 32 columns are two blocks of the row's four lanes
#pragma unroll
                    for (int j = 0; j < NBN; j += 2) {
                        float sum = 0.0f, m2 = 0.0f;
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum += y[j][e] + y[j + 1][e];
                        sum = halves32_sum(sum + __shfl_xor(sum, 16));
                        const float mu = sum * (1.0f / kNormGroup);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float a = y[j][e] - mu, b = y[j + 1][e] - mu;
                            m2 = fmaf(a, a, fmaf(b, b, m2));
                        }
                        m2 = halves32_sum(m2 + __shfl_xor(m2, 16));
                        const int n = n0 + wave_n * (BN / 2) + 16 * j;
                        if (g == 0 && m < M && n < N)
                            *reinterpret_cast<f32x2 *>(nf.out_stats + ((int64_t)m * (N / kNormGroup) + n / kNormGroup) * 2) = f32x2{sum, m2};
                    }
                }
            }
        };
        if (MODE == kNormAdd) {
            finish_norm(IntC<KERNL_ACT_NONE>());
            return;
        }
        switch (act) {
            case KERNL_ACT_RELU: finish_norm(IntC<KERNL_ACT_RELU>()); break;
            case KERNL_ACT_TANH: finish_norm(IntC<KERNL_ACT_TANH>()); break;
            case KERNL_ACT_GELU_ERF: finish_norm(IntC<KERNL_ACT_GELU_ERF>()); break;
            case KERNL_ACT_GELU_TANH: finish_norm(IntC<KERNL_ACT_GELU_TANH>()); break;
            case KERNL_ACT_SILU: finish_norm(IntC<KERNL_ACT_SILU>()); break;
            default: finish_norm(IntC<KERNL_ACT_NONE>()); break;
        }
        return;
    }

    // ---- epilogue: bias, optional pre-activation, activation, one rounding; 4 consecutive columns per lane and block
    const bool out_vec = out_cs == 1 && (out_rs & 3) == 0 && ((uintptr_t)out & 7) == 0;
    const bool ai_vec = act_in != nullptr && ai_cs == 1 && (ai_rs & 3) == 0 && ((uintptr_t)act_in & 7) == 0;
    // (the activation is chosen once, outside: a switch per element is a tree of scalar branches per element)
    auto finish = [&](auto act_c) __attribute__((always_inline)) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int i = 0; i < NBM; ++i) {
        const int m = m0 + wave_m * (BM / 2) + 16 * i + r;
#pragma unroll
        for (int j = 0; j < NBN; ++j) {
            const int n = n0 + wave_n * (BN / 2) + 16 * j + 4 * g;
            if (m >= M || n >= N) continue;
            float v[4], y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = acc[i][j][e] + bz[j][e];
                y[e] = apply_act16(v[e], ACT);
            }
            if (n + 4 <= N && out_vec) {
                const u32x2 p = {pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])};
                *reinterpret_cast<u32x2 *>(out + (int64_t)m * out_rs + n) = p;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) out[(int64_t)m * out_rs + (int64_t)(n + e) * out_cs] = from_float<T>(y[e]);
            }
            if (act_in != nullptr) {
                if (n + 4 <= N && ai_vec) {
                    const u32x2 p = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
                    *reinterpret_cast<u32x2 *>(act_in + (int64_t)m * ai_rs + n) = p;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < N) act_in[(int64_t)m * ai_rs + (int64_t)(n + e) * ai_cs] = from_float<T>(v[e]);
                }
            }
        }
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
}

// The same problem class with a LONG K (BERT-base's feed-forward down projection at batch 1: 128 x 768 x 3072): time per
// workgroup is latency x (bytes the workgroup pulls) / (bytes the CU keeps in flight), so the tiles get smaller still
// — 16 x 16 to 64 x 32, up to 256 workgroups — and the four waves no longer share a tile's k-tiles but deal them out:
// wave w multiplies k-tiles w, w + 4, ... of the WHOLE tile out of a ring of its own (no barrier in the loop, program
// order and the load counter are all the synchronisation), and the four partial tiles meet in LDS at the end.
// a wave's ring: 32 KB, 36 KB for the 12 KB stages of 64 x 32 tiles (three of them)
constexpr int small_ring_bytes(int bm, int bn, int waves) { return waves == 8 ? 16 * 1024 : (bm + bn) == 96 ? 36 * 1024 : 32 * 1024; }

template <typename T, int BM, int BN, int WAVES, int MODE>
__global__ void __launch_bounds__(64 * WAVES, 1)
linear_small_dealt_kernel(const T *__restrict__ X, const T *__restrict__ W, const T *__restrict__ bias,
                          T *__restrict__ out, T *__restrict__ act_in, int M, int N, int K, int64_t ldx, int64_t out_rs,
                          int64_t out_cs, int64_t ai_rs, int64_t ai_cs, int act, int tiles_m, NormFold nf) {
    typedef typename Vec8<T>::type vec8;
    constexpr int BK = 64, RB = BK * 2, CPR = BK / 8;
    static_assert(RB == SmallTileMap::ROW_BYTES && CPR == SmallTileMap::CHUNKS_PER_ROW, "tile rows as the tile map lays them out");
    constexpr int X_BYTES = BM * RB, W_BYTES = BN * RB, STAGE = X_BYTES + W_BYTES;
    constexpr int RING = small_ring_bytes(BM, BN, WAVES), S = RING / STAGE;  // a wave's ring and its stages
    constexpr int LX = BM * CPR / 64, LW = BN * CPR / 64, L = LX + LW;  // 1 KB loads per wave and stage
    constexpr int NBM = BM / 16, NBN = BN / 16;
    static_assert(S >= 3 && (S - 2) * L <= 63, "ring depth and wait count");
    static_assert(NBM * NBN * 1024 <= RING, "the partial tiles fit the rings");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    // tiles that share a weight tile (consecutive indices, the row tile running fastest) go to one XCD; with a single
    // row tile nothing is shared, and workgroups that run side by side had better read neighbouring weight rows
    const int tile = tiles_m > 1 ? xcd_contiguous_index((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;

    constexpr uint32_t kOutOfRange = 0x80000000u;
    const int rows_x = min(BM, M - m0), rows_w = min(BN, N - n0);
    const uint64_t xaddr = (uint64_t)(uintptr_t)(X + (int64_t)m0 * ldx);
    const uint64_t waddr = (uint64_t)(uintptr_t)(W + (int64_t)n0 * K);
    const u32x4 xrsrc = {(uint32_t)xaddr, (uint32_t)(xaddr >> 32) & 0xFFFFu,
                         (uint32_t)((((int64_t)rows_x - 1) * ldx + K) * 2), 0x00020000u};
    const u32x4 wrsrc = {(uint32_t)waddr, (uint32_t)(waddr >> 32) & 0xFFFFu, (uint32_t)((int64_t)rows_w * K * 2),
                         0x00020000u};
    // load i of the wave fills the 1 KB of 16-byte chunks [64 i, 64 i + 64) of an operand tile (the whole tile is the wave's)
    const int nk = (K + BK - 1) / BK;
    const int k_last = K - (nk - 1) * BK;
    uint32_t xd[LX], wd[LW], tail_bits = 0;
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int q = i * 64 + lane;
        const int row = SmallTileMap::load_row(q), c = SmallTileMap::load_chunk(q);
        xd[i] = row < rows_x ? (uint32_t)(((int64_t)row * ldx + c * 8) * 2) : kOutOfRange;
        if (c * 8 < k_last) tail_bits |= 1u << i;
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int q = i * 64 + lane;
        const int row = SmallTileMap::load_row(q), c = SmallTileMap::load_chunk(q);
        wd[i] = row < rows_w ? (uint32_t)(((int64_t)row * K + c * 8) * 2) : kOutOfRange;
        if (c * 8 < k_last) tail_bits |= 1u << (LX + i);
    }
    typedef __attribute__((address_space(3))) void lds_void;
    const uint32_t ring = (uint32_t)(uintptr_t)(lds_void *)smem + (uint32_t)wave * RING;
    auto load1 = [&](const u32x4 &rsrc, uint32_t off, uint32_t lds, int kbytes) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :: "s"(lds), "v"(off), "s"(rsrc), "s"(kbytes) : "memory", "m0");
    };
    // the wave's j-th k-tile (k-tile wave + 4 j of the problem) into stage `stage` of its ring
    // offsets clipped in place under a branch (as in the shared-tile kernel): to the chunks below K for the last k-tile
    // of the problem, to nothing at the wave's first request past it
    auto clip = [&](uint32_t keep) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");  // keeps this a branch: without it the compiler turns the block into selects
#pragma unroll
        for (int i = 0; i < LX; ++i) xd[i] = ((keep >> i) & 1u) != 0 ? xd[i] : kOutOfRange;
#pragma unroll
        for (int i = 0; i < LW; ++i) wd[i] = ((keep >> (LX + i)) & 1u) != 0 ? wd[i] : kOutOfRange;
    };
    auto request = [&](int j, int stage) __attribute__((always_inline)) {
        const int kt = wave + WAVES * j;
        if (kt >= nk - 1 && kt < nk + WAVES) clip(kt >= nk ? 0u : tail_bits);
        const uint32_t base = ring + (uint32_t)stage * STAGE;
        const int kbytes = kt < nk ? kt * BK * 2 : 0;
#pragma unroll
        for (int i = 0; i < LX; ++i) load1(xrsrc, xd[i], base + i * 1024, kbytes);
#pragma unroll
        for (int i = 0; i < LW; ++i) load1(wrsrc, wd[i], base + X_BYTES + i * 1024, kbytes);
    };
    int xoff[2][NBM], woff[2][NBN];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
        for (int i = 0; i < NBM; ++i) xoff[st][i] = SmallTileMap::frag_offset(16 * i + r, st, g);
#pragma unroll
        for (int j = 0; j < NBN; ++j) woff[st][j] = X_BYTES + SmallTileMap::frag_offset(16 * j + r, st, g);
    }
    f32x4_acc acc[NBM][NBN];
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) acc[i][j] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};

    // In the epilogue LPR = BN / 4 neighbouring lanes finish a row of the tile, 4 columns each: whole row pieces per store, and
    // a row's columns meet in neighbouring lanes (statistics).  What a thread needs of its row and columns is requested before
    // anything else.
    constexpr int LPR = BN / 4, ROWS = 64 * WAVES / LPR, OWN = (BM + ROWS - 1) / ROWS;
    const int own_row = tid / LPR, own_c = tid % LPR, n_own = n0 + 4 * own_c;
    auto lpr_sum = [](float v) __attribute__((always_inline)) { return LPR == 8 ? oct_sum(v) : quad_sum(v); };
    float bz[4];
    f32x4 cs = {0.0f, 0.0f, 0.0f, 0.0f};
    u32x2 res[OWN], gam = {0, 0}, bet = {0, 0};
    if (MODE == kNormApply) {  // (N is a multiple of 32 with a norm: every column of the tile exists)
        const f32x4 b32 = *reinterpret_cast<const f32x4 *>(nf.bias32 + n_own);
        cs = *reinterpret_cast<const f32x4 *>(nf.colsum + n_own);
#pragma unroll
        for (int e = 0; e < 4; ++e) bz[e] = b32[e];
    } else {
        load_bias4<T>(bias, n_own, N, ((uintptr_t)bias & 7) == 0, bz);
    }
    const bool row_stats = MODE == kNormApply || (MODE == kNormAdd && nf.in_stats != nullptr);
    if (MODE == kNormAdd) {
#pragma unroll
        for (int t = 0; t < OWN; ++t) {
            const int m = m0 + own_row + ROWS * t;
            res[t] = own_row + ROWS * t < rows_x ? *reinterpret_cast<const u32x2 *>(static_cast<const T *>(nf.residual) + (int64_t)m * nf.res_rs + n_own) : u32x2{0, 0};
        }
        if (row_stats) {
            gam = *reinterpret_cast<const u32x2 *>(static_cast<const T *>(nf.gamma) + n_own);
            if (nf.beta != nullptr) bet = *reinterpret_cast<const u32x2 *>(static_cast<const T *>(nf.beta) + n_own);
        }
    }
    if (MODE != kNormNone && row_stats)
        request_norm_stats<BM, WAVES>(nf, m0, rows_x, (uint32_t)(uintptr_t)(lds_void *)smem + WAVES * RING, wave, lane);
    const int mine = nk > wave ? (nk - wave + WAVES - 1) / WAVES : 0;  // k-tiles of this wave
#pragma unroll
    for (int j = 0; j < S - 1; ++j) request(j, j);
    int stage = 0;
    const unsigned char *my = smem + wave * RING;
    for (int j = 0; j < mine; ++j) {
        __builtin_amdgcn_s_waitcnt(0x0F70 | (((S - 2) * L) & 15) | ((((S - 2) * L) >> 4) << 14));
        const unsigned char *sb = my + stage * STAGE;
        vec8 xf[2][NBM], wf[2][NBN];
#pragma unroll
        for (int st = 0; st < 2; ++st) {
#pragma unroll
            for (int i = 0; i < NBM; ++i) xf[st][i] = *reinterpret_cast<const vec8 *>(sb + xoff[st][i]);
#pragma unroll
            for (int jj = 0; jj < NBN; ++jj) wf[st][jj] = *reinterpret_cast<const vec8 *>(sb + woff[st][jj]);
        }
        // the fragments are in registers before the stage is handed back to the loads
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        request(j + S - 1, stage == 0 ? S - 1 : stage - 1);
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < NBM; ++i)
#pragma unroll
                for (int jj = 0; jj < NBN; ++jj) acc[i][jj] = mfma16(wf[st][jj], xf[st][i], acc[i][jj]);
        stage = stage == S - 1 ? 0 : stage + 1;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the out-of-range requests of the last rounds are done with
    __syncthreads();                     // every ring is free: the partial tiles take their place

    // row statistics (staged behind the rings) merged by up to 16 threads a row, beside the stores of the partial tiles
    f32x2 *row_norm = reinterpret_cast<f32x2 *>(smem + WAVES * RING) - BM;  // (the end of the rings, which the partial tiles leave free)
    static_assert(WAVES * NBM * NBN * 1024 + BM * 8 <= WAVES * RING, "room behind the partial tiles");
    if (MODE != kNormNone && row_stats) {
        constexpr int SPAN = 64 * WAVES / BM < 16 ? 64 * WAVES / BM : 16, PER = norm_stats_bytes(BM) / BM / 8 / SPAN;
        const int row = tid / SPAN, c = tid % SPAN;
        if (row < BM) {
            const f32x2 *pairs = reinterpret_cast<const f32x2 *>(smem + WAVES * RING) + row * nf.in_groups;
            const float pivot = pairs[0][0] * nf.inv_group;
            NormMerge mg;
            auto merge = [&](int first, int last) __attribute__((always_inline)) {
                f32x2 v[PER];  // (read together: one after the other each costs an LDS round trip)
#pragma unroll
                for (int q = first; q < last; ++q) v[q] = pairs[SPAN * q + c < nf.in_groups ? SPAN * q + c : 0];
#pragma unroll
                for (int q = first; q < last; ++q)
                    if (SPAN * q + c < nf.in_groups) mg.take(v[q], pivot, nf.inv_group);
            };
            merge(0, PER / 2);
            if (SPAN * (PER / 2) < nf.in_groups) merge(PER / 2, PER);
            auto span_sum = [](float x) __attribute__((always_inline)) { return SPAN == 16 ? row16_sum(x) : SPAN == 8 ? oct_sum(x) : quad_sum(x); };
            mg.d = span_sum(mg.d);
            mg.dd = span_sum(mg.dd);
            mg.m2 = span_sum(mg.m2);
            if (c == 0) row_norm[row] = mg.finish(pivot, nf);
        }
    }
    float *red = reinterpret_cast<float *>(smem);  // [wave][block][lane][4]
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j)
            *reinterpret_cast<f32x4_acc *>(red + ((wave * (NBM * NBN) + i * NBN + j) * 64 + lane) * 4) = acc[i][j];
    __syncthreads();

    const bool out_vec = out_cs == 1 && (out_rs & 3) == 0 && ((uintptr_t)out & 7) == 0;
    const bool ai_vec = act_in != nullptr && ai_cs == 1 && (ai_rs & 3) == 0 && ((uintptr_t)act_in & 7) == 0;
    auto finish = [&](auto act_c) __attribute__((always_inline)) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int t = 0; t < OWN; ++t) {
        const int row = own_row + ROWS * t;
        if (BM < ROWS && row >= BM) break;
        // block (row / 16, own_c / 4), its lane (row % 16, own_c % 4)
        const int at = (((row >> 4) * NBN + (own_c >> 2)) * 64 + (own_c & 3) * 16 + (row & 15)) * 4;
        f32x4_acc sum = *reinterpret_cast<const f32x4_acc *>(red + at);
#pragma unroll
        for (int w = 1; w < WAVES; ++w) sum += *reinterpret_cast<const f32x4_acc *>(red + w * (NBM * NBN) * 256 + at);
        const int m = m0 + row, n = n_own;
        float pre[4], y[4], mean = 0.0f, rstd = 0.0f;
        if (MODE != kNormNone && row_stats) {
            const f32x2 norm = row_norm[row];
            mean = norm[0];
            rstd = norm[1];
        }
        if (MODE == kNormAdd) {
            float h[4], gm[4], bt[4];
            unpack4<T>(res[t], h);
            if (row_stats) {
                unpack4<T>(gam, gm);
                unpack4<T>(bet, bt);
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = fmaf((h[e] - mean) * rstd, gm[e], bt[e]);
            }
            float total = 0.0f, m2 = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = to_float(from_float<T>(sum[e] + bz[e] + h[e]));
                total += y[e];
            }
            // statistics of the stored values: the row's lanes, or with 16-column groups in 32-column tiles half of them
            const bool halves = LPR == 8 && nf.group == kNormGroupFew;
            const int cols = halves ? kNormGroupFew : BN;
            total = halves ? quad_sum(total) : lpr_sum(total);
            const float mu = total / (float)cols;
#pragma unroll
            for (int e = 0; e < 4; ++e) m2 = fmaf(y[e] - mu, y[e] - mu, m2);
            m2 = halves ? quad_sum(m2) : lpr_sum(m2);
            if (own_c % (cols / 4) == 0 && m < M)
                *reinterpret_cast<f32x2 *>(nf.out_stats + ((int64_t)m * (N / cols) + n_own / cols) * 2) = f32x2{total, m2};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pre[e] = MODE == kNormApply ? fmaf(fmaf(-mean, cs[e], sum[e]), rstd, bz[e]) : sum[e] + bz[e];
                y[e] = apply_act16(pre[e], ACT);
            }
        }
        if (m >= M || n >= N) continue;
        if (n + 4 <= N && out_vec) {
            const u32x2 p = {pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])};
            *reinterpret_cast<u32x2 *>(out + (int64_t)m * out_rs + n) = p;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < N) out[(int64_t)m * out_rs + (int64_t)(n + e) * out_cs] = from_float<T>(y[e]);
        }
        if (MODE == kNormNone && act_in != nullptr) {
            if (n + 4 <= N && ai_vec) {
                const u32x2 p = {pack2<T>(pre[0], pre[1]), pack2<T>(pre[2], pre[3])};
                *reinterpret_cast<u32x2 *>(act_in + (int64_t)m * ai_rs + n) = p;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) act_in[(int64_t)m * ai_rs + (int64_t)(n + e) * ai_cs] = from_float<T>(pre[e]);
            }
        }
    }
    };
    if (MODE == kNormAdd) {
        finish(IntC<KERNL_ACT_NONE>());
        return;
    }
    switch (act) {
        case KERNL_ACT_RELU: finish(IntC<KERNL_ACT_RELU>()); break;
        case KERNL_ACT_TANH: finish(IntC<KERNL_ACT_TANH>()); break;
        case KERNL_ACT_GELU_ERF: finish(IntC<KERNL_ACT_GELU_ERF>()); break;
        case KERNL_ACT_GELU_TANH: finish(IntC<KERNL_ACT_GELU_TANH>()); break;
        case KERNL_ACT_SILU: finish(IntC<KERNL_ACT_SILU>()); break;
        default: finish(IntC<KERNL_ACT_NONE>()); break;
    }
}

template <typename T, int BM, int BN, int WAVES, int MODE>
static void launch_small_dealt_mode(const LinearArgs &a, const NormFold &nf) {
    auto kern = linear_small_dealt_kernel<T, BM, BN, WAVES, MODE>;
    constexpr int LDS_BYTES = WAVES * small_ring_bytes(BM, BN, WAVES) + (MODE != kNormNone ? norm_stats_bytes(BM) : 0);
    static_assert(LDS_BYTES <= 160 * 1024, "one workgroup per CU");
    static bool attr_done = false;  // benign race: the attribute call is idempotent
    if (!attr_done) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
        attr_done = true;
    }
    const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
    hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * WAVES), LDS_BYTES, a.st, static_cast<const T *>(a.x),
                       static_cast<const T *>(a.w), static_cast<const T *>(a.bias), static_cast<T *>(a.out),
                       static_cast<T *>(a.act_in), a.M, a.N, a.K, a.x_rs, a.out_rs, a.out_cs, a.ai_rs, a.ai_cs, a.act,
                       tiles_m, nf);
}

template <typename T, int BM, int BN, int WAVES = 4>
static void launch_small_dealt(const LinearArgs &a, int mode, const NormFold &nf) {
    if (mode == kNormApply) launch_small_dealt_mode<T, BM, BN, WAVES, kNormApply>(a, nf);
    else if (mode == kNormAdd) launch_small_dealt_mode<T, BM, BN, WAVES, kNormAdd>(a, nf);
    else launch_small_dealt_mode<T, BM, BN, WAVES, kNormNone>(a, nf);
}

template <typename T>
static void run_small_dealt_t(const LinearArgs &a, int rows, int cols, int mode, const NormFold &nf) {
    if (cols == 16) {
        if (a.K >= 24 * 64) launch_small_dealt<T, 16, 16, 8>(a, mode, nf);  // three k-tiles a wave or more
        else launch_small_dealt<T, 16, 16>(a, mode, nf);
    } else if (rows == 16) launch_small_dealt<T, 16, 32>(a, mode, nf);
    else if (rows == 32) launch_small_dealt<T, 32, 32>(a, mode, nf);
    else launch_small_dealt<T, 64, 32>(a, mode, nf);
}

// rows x cols of a tile: 16 x 16, 16 x 32, 32 x 32 or 64 x 32
void run_small_dealt(const LinearArgs &a, int dtype, int rows, int cols, int mode, const NormFold &nf) {
    if (dtype == KERNL_F16) run_small_dealt_t<f16>(a, rows, cols, mode, nf);
    else run_small_dealt_t<bf16>(a, rows, cols, mode, nf);
}

template <typename T, int BM, int BN, int MODE>
static void launch_small_mode(const LinearArgs &a, const NormFold &nf) {
    auto kern = linear_small_kernel<T, BM, BN, MODE>;
    constexpr int LDS_BYTES = small_stages(BM, BN) * (BM + BN) * kSmallBK * 2 + (MODE != kNormNone ? norm_stats_bytes(BM) : 0);
    static bool attr_done = false;  // benign race: the attribute call is idempotent
    if (!attr_done) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
        attr_done = true;
    }
    const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
    hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(256), LDS_BYTES, a.st, static_cast<const T *>(a.x),
                       static_cast<const T *>(a.w), static_cast<const T *>(a.bias), static_cast<T *>(a.out),
                       static_cast<T *>(a.act_in), a.M, a.N, a.K, a.x_rs, a.out_rs, a.out_cs, a.ai_rs, a.ai_cs, a.act,
                       tiles_m, nf);
}

template <typename T, int BM, int BN>
static void launch_small(const LinearArgs &a, int mode, const NormFold &nf) {
    if (mode == kNormApply) launch_small_mode<T, BM, BN, kNormApply>(a, nf);
    else if (mode == kNormAdd) launch_small_mode<T, BM, BN, kNormAdd>(a, nf);
    else launch_small_mode<T, BM, BN, kNormNone>(a, nf);
}

// 32 x 64 tiles
void run_small(const LinearArgs &a, int dtype, int mode, const NormFold &nf) {
    if (dtype == KERNL_F16) launch_small<f16, 32, 64>(a, mode, nf);
    else launch_small<bf16, 32, 64>(a, mode, nf);
}

}  // namespace kernl
