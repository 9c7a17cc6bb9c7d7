// Linear layer for MIDDLING problems — 65 to some 3000 rows —, which give the big tile kernels less than a round of workgroups.
//
// What bounds such a launch: the tile loads of a CU.  It keeps some 32 KB of loads in flight however deep the ring is, so that they
// arrive at 32 KB per latency: 58 GB/s where the operands come from HBM, 110 from the memory-side cache, 140 from its L2 (a kernel
// that only loads, 256 workgroups; ring depths of 64 and 128 KB and every cache policy the same).  Loads of a line by several CUs at
// the same time wait the full latency each.  And where the waves that load also multiply, a full load path holds up their LDS reads
// and matrix instructions: 1024 x 768 x 3072 in 64 x 64 tiles took 15.5 us, the same with the loads alone 11.6, without them 8.9.  Hence
//   - waves that only load (four, behind those that multiply): what they wait for, nobody else waits for.  1024 x 768 x 3072
//     15.5 -> 13.0 us, 1024 x 3072 x 768 11.3 -> 9.8 in 128 x 128 tiles, 231 x 2304 x 768 6.6 -> 5.9;
//   - k-tiles dealt among the workgroups that share a weight or x tile (`turn`; see k_tiles_dealt in linear_kernels.h): 1024 x 4096 x 4096 in 128 x 128
//     tiles, weights from HBM, 39.6 -> 34.5 us, 512 x 12288 x 4096 in 256 x 128 tiles 54.7 -> 51, 333 x 22016 x 4096 in 192 x 192
//     tiles 66.5 -> 63; from the memory-side cache 1024 x 768 x 3072 12.5 -> 12.1, 231 x 768 x 3072 11.9 -> 11.2;
//   - tiles of 64 x 64 to 256 x 128, as large as still put a tile on (nearly) every CU: (BM + BN) x K bytes a tile;
//   - LDS fragments read one k-step ahead ACROSS the barrier (while k-step 1 of a k-tile is multiplied, k-step 0 of the next is read);
//     sched_barrier keeps the compiler from moving the reads back behind the multiplications;
//   - four multiplying waves of 32 x 32 in the 64 x 64 tile, two thirds of the LDS reads that eight of 16 x 32 need: 1024 x 768 x 3072 11.7 -> 10.9 us, 4096 x
//     768 x 3072 34.0 -> 32.3, 231 x 2304 x 768 5.7 -> 5.4.  (Larger tiles in four waves: 128 x 64 within 2 %, 128 x 128 9.1 -> 9.9 at K = 768.)
//   - the small tiles in rings of 64 to 72 KB, so that two workgroups share a CU where there are more tiles than CUs.
// Weight rows are placed in LDS so that a lane's blocks are consecutive output columns: 16-byte stores.
#include "linear_mid.h"

namespace kernl {

template <typename T, typename Cfg, bool GATED>
__global__ void __launch_bounds__(Cfg::WAVES * 64, Cfg::WAVES / 4)
linear_mid_kernel(const T *__restrict__ X, const T *__restrict__ W, const T *__restrict__ bias, T *__restrict__ out,
                  T *__restrict__ act_in, const float *__restrict__ row_scale, const T *__restrict__ residual, int M, int N, int K,
                  int64_t ldx, int64_t out_rs, int64_t out_cs, int64_t ai_rs, int64_t ai_cs, int64_t res_rs, int64_t res_cs, int act,
                  int tiles_m, MidGrid grid, float *__restrict__ part, int64_t part_rs, int range_kt) {
    linear_mid_tile<T, Cfg, GATED>(X, W, bias, out, act_in, row_scale, residual, M, N, K, ldx, out_rs, out_cs, ai_rs, ai_cs, res_rs, res_cs, act,
                                   tiles_m, grid, part, part_rs, range_kt, NoNorm());
}

template <typename T, typename Cfg, bool GATED>
static void launch_mid_cfg(const LinearArgs &a, const MidSplit &split = MidSplit()) {
    auto kern = linear_mid_kernel<T, Cfg, GATED>;
    static bool attr_done = false;  // benign race: the attribute call is idempotent
    if (!attr_done) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS);
        attr_done = true;
    }
    const int tiles_m = (a.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (a.N + Cfg::BN - 1) / Cfg::BN;
    MidGrid grid;
    const int blocks = mid_grid<Cfg>(tiles_m, tiles_n, split.splits, grid);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, (unsigned)split.splits), dim3(Cfg::WAVES * 64), Cfg::LDS, a.st, static_cast<const T *>(a.x),
                       static_cast<const T *>(a.w), static_cast<const T *>(a.bias), static_cast<T *>(a.out), static_cast<T *>(a.act_in),
                       a.row_scale, static_cast<const T *>(a.residual), a.M, a.N, a.K, a.x_rs, a.out_rs, a.out_cs, a.ai_rs, a.ai_cs,
                       a.res_rs, a.res_cs, a.act & (kGluBit - 1), tiles_m, grid, split.part, split.part_rs, split.range_kt);
}

template <typename T>
static int run_mid_t(const LinearArgs &a, int kind) {
    const bool gated = (a.act & kGluBit) != 0;
    switch (kind) {
        case 11: gated ? launch_mid_cfg<T, Mid64x64, true>(a) : launch_mid_cfg<T, Mid64x64, false>(a); return 1;
        case 15: gated ? launch_mid_cfg<T, Mid128x64, true>(a) : launch_mid_cfg<T, Mid128x64, false>(a); return 1;
        case 17: gated ? launch_mid_cfg<T, Mid128x128, true>(a) : launch_mid_cfg<T, Mid128x128, false>(a); return 1;
        case 18: gated ? launch_mid_cfg<T, Mid192x128, true>(a) : launch_mid_cfg<T, Mid192x128, false>(a); return 1;
        case 19: gated ? launch_mid_cfg<T, Mid192x192g, true>(a) : launch_mid_cfg<T, Mid192x192, false>(a); return 1;
        case 20: gated ? launch_mid_cfg<T, Mid128x256, true>(a) : launch_mid_cfg<T, Mid128x256, false>(a); return 1;
        case 21: gated ? launch_mid_cfg<T, Mid256x128, true>(a) : launch_mid_cfg<T, Mid256x128, false>(a); return 1;
        case 22:
            if (gated) return 0;
            launch_mid_cfg<T, Mid192x96, false>(a);
            return 1;
        default: return 0;
    }
}

int run_mid(const LinearArgs &a, int dtype, int kind) { return dtype == KERNL_F16 ? run_mid_t<f16>(a, kind) : run_mid_t<bf16>(a, kind); }

// ranges of K: no gates (the value of the gate is not linear in the sums), and tiles whose partial results pay
template <typename T>
static void run_mid_split_t(const LinearArgs &a, int tile, const MidSplit &split) {
    switch (tile) {
        case 11: launch_mid_cfg<T, Mid64x64, false>(a, split); break;
        case 15: launch_mid_cfg<T, Mid128x64, false>(a, split); break;
        case 18: launch_mid_cfg<T, Mid192x128, false>(a, split); break;
        case 22: launch_mid_cfg<T, Mid192x96, false>(a, split); break;
        default: launch_mid_cfg<T, Mid128x128, false>(a, split); break;
    }
}

void run_mid_split(const LinearArgs &a, int dtype, int tile, const MidSplit &split) {
    if (dtype == KERNL_F16) run_mid_split_t<f16>(a, tile, split);
    else run_mid_split_t<bf16>(a, tile, split);
}

}  // namespace kernl
