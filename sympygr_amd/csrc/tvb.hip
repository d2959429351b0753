// The kernels of one_pass.h that add TVB dissipation to a finished right-hand
// side or RK stage (BSSN): k_rhs runs with sigma 0, this pass reads every halo
// tile once more and adds sigma (D_x + D_y + D_z).  Only halo tiles in LDS: two
// workgroups per CU fit with 8^3 tiles (128 registers; the general shapes take
// 170 and run one).  64 blocks of 32^3 points with flagged faces, TVB5: the whole
// call 2.59 -> 1.89 ms, 0.7 of it here (each tap from global memory instead of LDS,
// the pass took 0.95).  TVB3 takes as long: memory traffic, not the forms.
#include "one_pass.h"

namespace sgr {

template <Pass PASS, bool GEN, bool RK>
__global__ __launch_bounds__(512, GEN ? 2 : 4) void k_tvb_add(FieldPtrs in, OutPtrs out, const BlockDesc *__restrict__ blocks,
                                                    const uint32_t *__restrict__ tile_block,
                                                    const uint32_t *__restrict__ order, RkArgs rk, TileRanges ranges,
                                                    TvbArgs tv)
{
    one_pass<PASS, false, GEN, RK, false>(in, out, blocks, tile_block, order, Params{}, rk, ranges, tv);
}

template <Pass PASS, bool GEN, bool RK>
static hipError_t launch_list(const LaunchArgs &a, const TileList &l, hipEvent_t e0, hipEvent_t e1, hipStream_t s)
{
    TileRanges r;
    const uint32_t grid = list_grid(l, GEN ? a.grid_cap : 2 * a.grid_cap, r);
    hipExtLaunchKernelGGL((k_tvb_add<PASS, GEN, RK>), dim3(grid), dim3(512), 0, s, e0, e1, 0, a.in, a.out, a.blocks,
                          a.tile_block, l.order, a.rk, r, TvbArgs{a.lam, a.lam_span, a.diss_sigma});
    return hipGetLastError();
}

template <Pass PASS, bool RK>
static hipError_t launch_lists(const LaunchArgs &a, hipStream_t s)
{
    const bool fast = a.list[0].lo[8] > a.list[0].lo[0], gen = a.list[1].lo[8] > a.list[1].lo[0];
    hipError_t e = hipSuccess;
    if (fast) e = launch_list<PASS, false, RK>(a, a.list[0], a.ev[2], gen ? nullptr : a.ev[3], s);
    if (e == hipSuccess && gen) e = launch_list<PASS, true, RK>(a, a.list[1], fast ? nullptr : a.ev[2], a.ev[3], s);
    return e;
}

hipError_t launch_tvb(const LaunchArgs &a, hipStream_t s)
{
    if (a.diss == 2)
        return a.rk.stage >= 0 ? launch_lists<Pass::TVB5, true>(a, s) : launch_lists<Pass::TVB5, false>(a, s);
    return a.rk.stage >= 0 ? launch_lists<Pass::TVB3, true>(a, s) : launch_lists<Pass::TVB3, false>(a, s);
}

}  // namespace sgr
