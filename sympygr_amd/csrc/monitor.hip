// The kernels of one_pass.h that evaluate the constraints and Psi4: 17 fields,
// seven with second derivatives, each halo tile read once and nothing staged in
// memory.  The derivative pass and the pointwise pass that they replace moved
// about 140 staged values per point both ways.  216 blocks of 32^3 interior
// points, FP64, with Psi4: 4.35 -> 1.84 ms.  ROUND: mixed-precision plans, whose
// staged derivatives are float.
#include "one_pass.h"

namespace sgr {

template <bool PSI4, bool GEN, bool ROUND>
__global__ __launch_bounds__(512, 2) void k_monitor(FieldPtrs in, OutPtrs out, const BlockDesc *__restrict__ blocks,
                                                    const uint32_t *__restrict__ tile_block,
                                                    const uint32_t *__restrict__ order, TileRanges ranges)
{
    one_pass<PSI4 ? Pass::PSI4 : Pass::CONSTRAINTS, false, GEN, false, ROUND>(in, out, blocks, tile_block, order, Params{},
                                                                              RkArgs{}, ranges);
}

template <bool PSI4, bool GEN, bool ROUND>
static hipError_t launch_list(const LaunchArgs &a, const OutPtrs &out, const TileList &l, hipStream_t s)
{
    TileRanges r;
    const uint32_t grid = list_grid(l, a.grid_cap, r);
    hipLaunchKernelGGL((k_monitor<PSI4, GEN, ROUND>), dim3(grid), dim3(512), 0, s, a.in, out,
                       a.blocks, a.tile_block, l.order, r);
    return hipGetLastError();
}

template <bool PSI4, bool ROUND>
static hipError_t launch_lists(const LaunchArgs &a, const OutPtrs &out, hipStream_t s)
{
    hipError_t e = hipSuccess;
    if (a.list[0].lo[8] > a.list[0].lo[0]) e = launch_list<PSI4, false, ROUND>(a, out, a.list[0], s);
    if (e == hipSuccess && a.list[1].lo[8] > a.list[1].lo[0]) e = launch_list<PSI4, true, ROUND>(a, out, a.list[1], s);
    return e;
}

hipError_t launch_monitor(const LaunchArgs &a, const OutPtrs &out, bool psi4, hipStream_t s)
{
    if (a.mixed) return psi4 ? launch_lists<true, true>(a, out, s) : launch_lists<false, true>(a, out, s);
    return psi4 ? launch_lists<true, false>(a, out, s) : launch_lists<false, false>(a, out, s);
}

}  // namespace sgr
