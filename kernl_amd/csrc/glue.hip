// The glue around a captured model's kernels, where a launch (1.6 us in a graph, 3 to 4 in front of one) outweighs the work:
// copies of the call's inputs into the static buffers, and padding masks as additive masks.
#include "common.h"

namespace kernl {

constexpr int kCopyMax = 8;
struct CopyList {
    const u32x4 *src[kCopyMax];
    u32x4 *dst[kCopyMax];
    int64_t bytes[kCopyMax];
    int first_block[kCopyMax + 1];  // blocks of list entry i: first_block[i] .. first_block[i + 1] - 1
};
constexpr int kCopyBlockBytes = 256 * 16 * 4;

// One launch for all of a call's inputs.  A block owns 16 KB of one of them: four 16-byte pieces per thread, all requested before
// any is stored.
__global__ void __launch_bounds__(256) copy_many_kernel(CopyList list, int n) {
    const int block = blockIdx.x;
    int i = 0;
    while (i + 1 < n && block >= list.first_block[i + 1]) ++i;
    const int64_t base = (int64_t)(block - list.first_block[i]) * kCopyBlockBytes;
    const int64_t left = list.bytes[i] - base;
    const u32x4 *src = list.src[i] + base / 16;
    u32x4 *dst = list.dst[i] + base / 16;
    const int whole = (int)((left < kCopyBlockBytes ? left : kCopyBlockBytes) / 16), t = threadIdx.x;
    u32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (t + 256 * k < whole) v[k] = src[t + 256 * k];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (t + 256 * k < whole) dst[t + 256 * k] = v[k];
    const int64_t tail = left - (int64_t)whole * 16;
    if (left < kCopyBlockBytes && t < tail)
        reinterpret_cast<unsigned char *>(dst + whole)[t] = reinterpret_cast<const unsigned char *>(src + whole)[t];
}

// out[i] = mask[i] != 0 ? on : off
template <typename M, typename T>
__global__ void __launch_bounds__(256) select_mask_kernel(const M *__restrict__ mask, T *__restrict__ out, int64_t n, float on, float off) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = from_float<T>(mask[i] != 0 ? on : off);
}

template <typename M>
static void launch_select(const void *mask, void *out, int64_t n, float on, float off, int dtype, hipStream_t st) {
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    const M *m = static_cast<const M *>(mask);
    if (dtype == KERNL_F16) hipLaunchKernelGGL((select_mask_kernel<M, f16>), grid, block, 0, st, m, static_cast<f16 *>(out), n, on, off);
    else if (dtype == KERNL_BF16) hipLaunchKernelGGL((select_mask_kernel<M, bf16>), grid, block, 0, st, m, static_cast<bf16 *>(out), n, on, off);
    else hipLaunchKernelGGL((select_mask_kernel<M, float>), grid, block, 0, st, m, static_cast<float *>(out), n, on, off);
}

}  // namespace kernl

extern "C" int kernl_copy_many(int count, const void *const *src, void *const *dst, const int64_t *bytes, void *stream) {
    using namespace kernl;
    if (count < 0 || count > kCopyMax || (count > 0 && (src == nullptr || dst == nullptr || bytes == nullptr)))
        return set_error(KERNL_ERR_INVALID_ARG, "copy_many: 0 to %d pieces", kCopyMax);
    CopyList list = {};
    int n = 0;
    int64_t blocks = 0;
    for (int i = 0; i < count; ++i) {
        if (bytes[i] < 0 || (bytes[i] > 0 && (src[i] == nullptr || dst[i] == nullptr)))
            return set_error(KERNL_ERR_INVALID_ARG, "copy_many: piece %d has a NULL pointer or a negative size", i);
        if (bytes[i] == 0) continue;
        if (!aligned16(src[i]) || !aligned16(dst[i])) return set_error(KERNL_ERR_UNSUPPORTED, "copy_many: pieces must be 16-byte aligned");
        list.src[n] = static_cast<const u32x4 *>(src[i]);
        list.dst[n] = static_cast<u32x4 *>(dst[i]);
        list.bytes[n] = bytes[i];
        list.first_block[n++] = (int)blocks;
        blocks += (bytes[i] + kCopyBlockBytes - 1) / kCopyBlockBytes;
        if (blocks > INT32_MAX) return set_error(KERNL_ERR_UNSUPPORTED, "copy_many: too many bytes");
        list.first_block[n] = (int)blocks;
    }
    if (n == 0) return KERNL_OK;
    hipLaunchKernelGGL(copy_many_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), list, n);
    return check_launch("copy_many");
}

extern "C" int kernl_select_mask_fwd(const void *mask, int mask_bytes, float on, float off, void *out, int64_t n, int dtype, void *stream) {
    using namespace kernl;
    if (n < 0 || (n > 0 && (mask == nullptr || out == nullptr))) return set_error(KERNL_ERR_INVALID_ARG, "select_mask: mask and out must not be NULL");
    if (mask_bytes != 1 && mask_bytes != 4 && mask_bytes != 8) return set_error(KERNL_ERR_UNSUPPORTED, "select_mask: mask elements of 1, 4 or 8 bytes");
    if (dtype != KERNL_F16 && dtype != KERNL_BF16 && dtype != KERNL_F32) return set_error(KERNL_ERR_UNSUPPORTED, "select_mask: unknown dtype %d", dtype);
    if (n > (int64_t)INT32_MAX * 128) return set_error(KERNL_ERR_UNSUPPORTED, "select_mask: too many elements");
    if (n == 0) return KERNL_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (mask_bytes == 1) launch_select<uint8_t>(mask, out, n, on, off, dtype, st);
    else if (mask_bytes == 4) launch_select<int32_t>(mask, out, n, on, off, dtype, st);
    else launch_select<int64_t>(mask, out, n, on, off, dtype, st);
    return check_launch("select_mask");
}
