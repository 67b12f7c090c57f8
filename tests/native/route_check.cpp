// Which form plan_contraction gives a contraction, for tests on the CPU.
#include "../../jet_amd/csrc/contract_plan.hpp"

using namespace jet_hip;

// out: form (0 product, 1 fused pass in place, 2 short k in place, 3 few outputs
// in place), kernel, launches, slices, and the workspace's bytes.
extern "C" int contraction_route(int mode, int ra, const int32_t *ma, const int64_t *ea, int rb,
                                 const int32_t *mb, const int64_t *eb, int rc, const int32_t *mc,
                                 int64_t *out)
{
    const ContractionDesc d =
        plan_contraction(mode == 2 ? 16 : 8, mode, 0, ra, ma, ea, rb, mb, eb, rc, mc);
    out[0] = d.fused_small ? 1 : d.stream_shortk ? 2 : d.stream_dot ? 3 : 0;
    out[1] = d.gemm_kernel;
    const bool split = d.gemm_kernel == kGemmBf16x3 || d.gemm_kernel == kGemmBf16x4m ||
                       d.gemm_kernel == kGemmF16x4m;
    out[2] = out[0] == 1 || out[0] == 2 ? 1
             : out[0] == 3              ? 2
                                        : 1 + (d.need_a && !d.fuse_a) + (d.need_b && !d.fuse_b) +
                                 d.need_c + (split ? 2 : 0) + (d.gemm_kernel == kGemmSplitK) +
                                 (d.chunks > 1 || d.slices > 1);
    out[3] = d.slices;
    out[4] = (int64_t)d.workspace;
    return 0;
}

// Tiles of the form that an FP32 (aligned rows or not) or FP64 product takes.
extern "C" int64_t product_tiles(int fp64, int aligned, int64_t M, int64_t N, int64_t K)
{
    int form = 0;
    const TileForm *f = fp64 ? kF64Forms : aligned ? kF32x6Forms : kF32x6DwordForms;
    (void)(fp64      ? tile_time(kF64Forms, M, N, K, 1, &form)
           : aligned ? tile_time(kF32x6Forms, M, N, K, 1, &form)
                     : tile_time(kF32x6DwordForms, M, N, K, 1, &form));
    return ceil_div(M, f[form].bm) * ceil_div(N, f[form].bn);
}
