// Definitions shared by the attention kernels (attention.hip, attention_pipe.hip): parameter block, mask helpers.
#pragma once

#include <math.h>

#include <type_traits>

#include "common.h"

namespace kernl {

static constexpr float kLog2eA = 1.4426950408889634f;
static constexpr float kNegBig = -1.0e30f;            // anything below: exp2(x - rowmax) is exactly 0
static constexpr float kClampFloor = -1.7014118e38f;  // scaled mask values are kept finite (-FLT_MAX / 2)
static constexpr float kRescaleThreshold = 8.0f;  // log2 units
static constexpr float kMaskedScore = -32768.0f;  // base-2 scores below this are mask values, not scores
// A mask value (base-2 domain) at or below this marks a dead key: added to any score a 16-bit model produces it stays
// below kMaskedScore, so the key weighs exactly 0 in every row that has an ordinary key, and a key tile of dead keys only
// is not visited at all.  -inf and the fp32 / bf16 "minimum" masks are far below it, and so is the fp16 one that models
// build in their own dtype (finfo(float16).min = -65504, -94505 in the base-2 domain) — which kNegBig does not catch.
static constexpr float kDeadMask = 2.0f * kMaskedScore;

enum { MASK_NONE = 0, MASK_VECTOR = 1, MASK_MATRIX = 2 };

struct AttnParams {
    const void *q, *k, *v, *mask;
    void *o;
    int B, H, M, N;
    int64_t qs[4], ks[4], vs[4], os[4];  // element strides {batch, head, row, col}
    int64_t ms[4];                       // mask strides, 0 on broadcast dims
    int mask_dtype;
    float scale_log2;  // sm_scale * log2(e)
    float sm_scale;
    float clamp;  // replacement for -inf mask entries
    int nq_tiles;
    int mask_fast;  // matrix mask rows: 1 = readable as aligned 4-element vectors through 32-bit offsets,
                    // 2 = 16-byte chunks of a row are aligned too (they can be staged through LDS)
    int16_t xcd_by_batch;  // workgroups of one batch entry (all heads) share an XCD instead of those of one head
    int16_t rank_group;    // causal: heads whose tiles are ranked together (ranked_item)
    int causal_off;  // causal: query row m sees keys 0 .. m + causal_off (0: top-left aligned)
};
// With the argument behind it attention_short.hip's arguments end inside four lines; a fifth costs the smallest launches 0.25 of 3.1 us.
static_assert(sizeof(AttnParams) <= 248, "kernel arguments");

__device__ __forceinline__ float load_mask_value(const void *mask, int dtype, int64_t off) {
    if (dtype == KERNL_F32) return static_cast<const float *>(mask)[off];
    if (dtype == KERNL_F16) return (float)static_cast<const f16 *>(mask)[off];
    return (float)static_cast<const bf16 *>(mask)[off];
}

// mask value -> additive term in the log2 domain, finite.
__device__ __forceinline__ float scale_mask(float mv, float clamp) {
    if (mv == -INFINITY) mv = clamp;
    return fmaxf(mv * kLog2eA, kClampFloor);
}


// How attention_short.hip and attention_split.hip place value rows in LDS: the row's 16-byte chunk c at c ^ value_flip(row).  A transposing
// read takes 8 bytes from each of 8 rows at 4 places a quarter of a row apart; rows of head size 64 alternate between the halves of the
// banks, so one bit of the row spreads the rest, rows of head size 128 need two (with one bit: 4 lanes to a bank instead of 2).
template <int D>
__host__ __device__ static inline int value_flip(int row) {
    return D == 64 ? (row >> 1) & 1 : row & 3;
}

// Software-pipelined MFMA kernel (attention_pipe.hip).  Handles head sizes 64 and 128 with no mask or with a per-key
// mask of at most kPipeMaxMaskKeys keys (non-causal), and causal attention without a mask.  Taken without
// causality at head size 64, from kPipeMinKeys keys on and for small grids; causal grids by pipe_pays_causal (attention_pipe.hip); or whenever it
// applies, with `force`.  Returns false when it does not take the problem.
static constexpr int kPipeMaxMaskKeys = 2048;
static constexpr int kPipeMinKeys = 1024;
bool launch_attention_pipe(const AttnParams &p, int D, int dtype, int mask_mode, bool causal, bool force, hipStream_t st);

// Kernel for short key sequences (attention_short.hip): up to kShortMaxKeys keys, no mask or a per-key mask, causal or not.
static constexpr int kShortMaxKeys = 256;
// Where it is the fastest (graph replay, us, before -> with it; [batch, heads, keys, head size], per-key mask unless said):
//   [1,12,16,64] 4.8 -> 2.6   [3,12,77,64] 6.1 -> 3.4   [8,12,128,64] 6.0 -> 3.9   [32,12,128,64] 7.8 -> 5.9   [4,12,256,64] 7.6 -> 5.1
//   [512,12,16,64] 40 -> 10.6   [1,32,128,128] causal 7.4 -> 5.1   [4,16,256,128] 10.7 -> 8.5   [64,32,30,128] 26 -> 12.8
// Every wave reads all keys of its head from LDS, so with enough workgroups to fill the chip several times over the kernels
// whose waves share 128-row tiles win: [64,12,128,64] 12.3 -> 12.3, [16,12,256,64] 8.5 -> 9.6 without a mask, [8,32,160,128] 15.0
// -> 17.6.  The limits lie at the last grid of each size where it was ahead with and without a mask.
// Many query rows over few keys (cross-attention) stage keys and values once per 64 rows, where the other kernels do per 128.  Up to
// 32 keys that is little (at worst [1,8,8192,128] over 16 keys 10.7 -> 11.0 without a mask, 12.0 -> 11.4 with one), and a mask costs
// the others its classification ([16,16,8192,64] over 64 keys 150 -> 133); without one and beyond 32 keys they win from some grid on:
// head size 128, 33 to 64 keys: 128 workgroups 5.8 -> 4.8, 192 5.9 -> 5.1, 512 7.1 -> 7.9, 1024 9.8 -> 11.5; head size 64: 16384
// workgroups 59 -> 46, 32768 124 -> 133.  Up to 64 rows their 128-row tiles are half empty.
static inline bool attention_short_pays(int64_t workgroups, int64_t M, int N, int D, bool masked) {
    if (N <= 32 || (N <= 64 && (masked || M <= 64))) return true;
    if (N <= 64) return workgroups <= (D == 64 ? 16384 : 384);
    if (D == 64) return workgroups <= (N <= 128 ? 1024 : N <= 192 ? 512 : 384);
    return workgroups <= (N <= 128 ? 384 : 256);
}
// Kernel whose waves split every key tile (attention_split.hip): causal, no mask; workgroups of 64 rows.
void run_attention_split(const AttnParams &p, int D, int dtype, hipStream_t st);
// Where it is the fastest: as long as its workgroups, one a CU, are one round.  Beyond that the last to start are the shortest (the longest
// go first), and with many tiles a head these still fit in behind; with few, or where new rows over a cache make all of them long, they do
// not (us, pipelined or streaming kernel -> this one, [heads, rows, head size]: [48,333,128] 288 workgroups 11.3 -> 13.3; [24,700,128] 264
// 15.6 -> 14.0; [32,700,128] 352 16.8 -> 17.3; [16,1111,128] 288 20.7 -> 18.4; [24,1024,128] 384 20.3 -> 21.1; [12,2048,128] 384 33.7 ->
// 30.9; 300 rows over 1024 keys, 64 heads, 320 workgroups 23.8 -> 31.6).  At head size 64 the pipelined kernel is level from some 512 keys
// on and ahead later ([32,333,64] 8.0 -> 7.6, [32,512,64] 9.1 -> 9.0, [24,1000,64] 12.5 -> 14.6); up to kShortMaxKeys keys
// attention_short.hip is ahead by a fifth.
static inline bool attention_split_pays(int64_t heads, int64_t M, int64_t N, int64_t start, int D) {
    if (N <= kShortMaxKeys || (D == 64 && N > 512)) return false;
    const int64_t tiles = (M + 63) / 64, behind = tiles >= 11 && start * 4 <= M ? 4 * tiles : 0;
    return heads * tiles <= 256 + (behind < 128 ? behind : 128);
}
void run_attention_short(const AttnParams &p, int D, int dtype, bool masked, bool causal, hipStream_t st);

}  // namespace kernl
