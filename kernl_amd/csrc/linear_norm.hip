// linear + residual + LayerNorm in one launch: which shapes take it, and its C entry points.
#include "linear_kernels.h"
#include "norm_exchange.h"

namespace kernl {

// The tiles it runs on, smallest first, by the hook's values (12 .. 14 dealt k-tiles, 5 and 6 the wide kernel, the others tiles of linear_mid.h),
// and the threads that hold a tile's results.
struct NormTile {
    int kind, bm, bn, threads;
};
static constexpr NormTile kNormTiles[] = {{12, 16, 32, 128}, {13, 32, 32, 256}, {14, 64, 32, 512}, {11, 64, 64, 256}, {15, 128, 64, 512},
                                          {17, 128, 128, 512}, {18, 192, 128, 512}, {20, 128, 256, 512}, {21, 256, 128, 512}, {19, 192, 192, 512},
                                          {6, 256, 192, 256}, {5, 256, 256, 256}};

// The smallest tile of which one round covers the rows: all workgroups of a row have to run at the same time, and smaller tiles
// are faster as long as they do.  us, this launch / what ran before it (product and add + LayerNorm, or K split with the LayerNorm in its second
// launch), one process, weights in the memory-side cache:
//   rows     768 x 768      768 x 3072     1024 x 1024    512 x 2048
//    128     5.4 /  6.6     7.1 /  8.2     5.9 /  7.2     6.2 /  6.8
//    256     6.2 /  7.2     8.0 /  9.3     6.7 /  7.2     6.6 /  7.5
//   1024     7.5 /  9.0    13.2 / 15.0     8.3 /  9.7    10.1 / 11.6
//   2048     9.4 / 11.1    19.9 / 21.6    11.4 / 12.8    10.7 / 13.0
//   4096    12.1 / 17.7    26.2 / 29.1    16.0 / 22.0    16.4 / 18.4
//   8192    19.2 / 22.5    42.8 / 44.1    25.7 / 30.1    23.4 / 30.1
//  12288    26.0 / 30.2    56.1 / 63.4    39.2 / 47.9    31.3 / 35.7
//  14000    29.5 / 33.2    65.0 / 69.9                                   (from here on, and 1024 columns beyond 8192 rows, the wide kernel: 256 x 192
//  16384    30.8 / 36.4    69.6 / 74.4    42.2 / 57.8                     tiles, or 256 x 256; 16384 x 1024 x 4096 108.9 / 123.9)
//  20000    35.9 / 49.4    84.0 / 102.9   (two rounds)   (24000) 55.3 / 68.9
// Left to the others: weights that come from HBM (not measured); a K beyond 2048 where 32-row tiles no longer do and 64 x 64 leave the chip half
// empty, which is where K split wins (512 x 768 x 3072 12.0 / 11.2, 600 rows 12.6 / 11.8, 682 12.8 / 13.3; 682 x 1024 x 4096 16.8 / 16.6, 800
// rows 17.2 / 17.9).
static const NormTile *norm_tile(int64_t M, int64_t N, int64_t K) {
    for (const NormTile &t : kNormTiles) {
        const int64_t tiles_n = N / t.bn, tiles = (M + t.bm - 1) / t.bm * tiles_n;
        if (N % t.bn != 0 || tiles_n > exchange_most(exchange_lanes(t.bm, t.threads))) continue;
        if (g_linear_force_tile != 0) {
            if (t.kind == g_linear_force_tile) return &t;
            continue;
        }
        if (tiles > 256) continue;
        // (the larger ones over more than 1024 columns, 600 x 2048 x 2048 16.8 against 16.2 and 800 x 1536 x 1536 15.5 against 13.3, and 128 x 64 tiles over a
        // long K that leave a third of the chip empty, 1365 x 768 x 3072 20.7 against 19.8, 1365 x 1024 x 4096 27.2 against 26.3, are slower)
        if (N > 1024 && t.bm * t.bn > 64 * 64) return nullptr;
        if (t.kind == 15 && K > 2048 && tiles < (K <= 3072 ? 160 : 208)) return nullptr;
        // 64 x 32 tiles with dealt k-tiles: 682 x 512 x 2048 8.7 against 10.1 in 64 x 64, 1024 rows (a full round) 10.6 against 10.1, 682 x 768 x 768 7.6
        // against 7.5
        if (t.kind == 14 && (K < 1536 || K > 2048 || tiles > 208)) continue;
        return t.kind != 11 || K <= 2048 || tiles >= (K <= 3072 ? 128 : 200) ? &t : nullptr;
    }
    return nullptr;
}

}  // namespace kernl

extern "C" int64_t kernl_linear_exchange_bytes(int64_t M, int64_t N, int64_t K) {
    using namespace kernl;
    if (M <= 64 || N < 128 || K < 64 || M > INT32_MAX || K >= (1 << 22) || K % 8 != 0 || !weight_cached(N, K)) return 0;
    const NormTile *t = norm_tile(M, N, K);
    return t != nullptr ? exchange_words((M + t->bm - 1) / t->bm, N / t->bn, t->bm) * 8 : 0;
}

extern "C" int kernl_linear_add_norm_fwd(const void *x, const void *w, const void *bias, const void *residual, const void *gamma, const void *beta,
                                         float eps, void *out, float *sums, void *region, void *next_region, int64_t region_bytes, int patience,
                                         int64_t M, int64_t N, int64_t K, int64_t x_rs, int64_t res_rs, int64_t out_rs, int dtype, void *stream) {
    using namespace kernl;
    if (x == nullptr || w == nullptr || residual == nullptr || gamma == nullptr || out == nullptr || sums == nullptr || region == nullptr || next_region == nullptr)
        return set_error(KERNL_ERR_INVALID_ARG, "linear + add + LayerNorm: x, w, residual, gamma, out, sums and both regions must not be NULL");
    if (M <= 0 || N <= 0 || K <= 0 || region_bytes < 0)
        return set_error(KERNL_ERR_INVALID_ARG, "linear + add + LayerNorm: bad sizes M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
    if (dtype != KERNL_F16 && dtype != KERNL_BF16)
        return set_error(KERNL_ERR_UNSUPPORTED, "linear + add + LayerNorm: only f16 and bf16 are supported, got dtype %d", dtype);
    const int64_t need = kernl_linear_exchange_bytes(M, N, K);
    if (need == 0)
        return set_error(KERNL_ERR_UNSUPPORTED, "linear + add + LayerNorm: M=%lld N=%lld K=%lld is faster in two launches (kernl_linear_exchange_bytes "
                         "returns 0)", (long long)M, (long long)N, (long long)K);
    auto aligned8 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; };
    if (x_rs >= (1 << 22) || x_rs % 8 != 0 || x_rs < K || !aligned16(x) || !aligned16(w) || res_rs % 4 != 0 || out_rs % 8 != 0 || !aligned8(bias) ||
        !aligned8(residual) || !aligned8(gamma) || !aligned8(beta) || !aligned16(out) || !aligned16(sums))
        return set_error(KERNL_ERR_UNSUPPORTED, "linear + add + LayerNorm: K must be a multiple of 8, x, w, out and sums 16-byte aligned with 16-byte "
                         "aligned rows, everything else 8-byte aligned");
    if (region_bytes < need || region_bytes % 8 != 0 || region_bytes > INT32_MAX || !aligned8(region) || !aligned8(next_region))
        return set_error(KERNL_ERR_INVALID_ARG, "linear + add + LayerNorm: each region must hold %lld bytes, 8-byte aligned", (long long)need);
    LinearArgs a;
    a.x = x; a.w = w; a.bias = bias; a.out = out; a.act_in = nullptr;
    a.M = (int)M; a.N = (int)N; a.K = (int)K;
    a.x_rs = x_rs; a.x_cs = 1;
    a.out_rs = out_rs; a.out_cs = 1;
    a.ai_rs = a.ai_cs = 0;
    a.act = KERNL_ACT_NONE;
    a.st = static_cast<hipStream_t>(stream);
    NormExchange nx;
    nx.residual = residual; nx.res_rs = res_rs;
    nx.gamma = gamma; nx.beta = beta; nx.eps = eps;
    nx.words = static_cast<uint64_t *>(region);
    nx.clear = static_cast<uint64_t *>(next_region);
    nx.clear_words = (int)(region_bytes / 8);
    if (patience >= 0) nx.patience = patience;
    nx.sums = sums;
    nx.inv_n = 1.0f / (float)N;
    const NormTile *t = norm_tile(M, N, K);
    if (t->kind >= 12 && t->kind <= 14) run_small_dealt_norm(a, dtype, t->bm, nx);
    else if (t->kind == 5 || t->kind == 6) run_wide_norm(a, dtype, t->bn, nx);
    else run_mid_norm(a, dtype, t->kind, nx);
    return check_launch("linear + add + LayerNorm");
}
