// The kernels of one_pass.h that evaluate the BSSN right-hand side.
#include "one_pass.h"

namespace sgr {

template <bool UPWIND, bool GEN, bool RK>
__global__ __launch_bounds__(512, 2) void k_rhs(FieldPtrs in, OutPtrs out, const BlockDesc *__restrict__ blocks,
                                                const uint32_t *__restrict__ tile_block,
                                                const uint32_t *__restrict__ order, Params P, RkArgs rk, uint32_t tile0,
                                                TileRanges ranges)
{
    one_pass<Pass::BSSN, UPWIND, GEN, RK, false>(in, out, blocks, tile_block, order, P, rk, tile0, ranges);
}

// k_rhs over one list of tiles: at most one workgroup per CU, a multiple of 8
// so that every XCD's range is served.
template <bool UPWIND, bool GEN, bool RK>
static hipError_t launch_list(const LaunchArgs &a, const TileList &l, hipEvent_t e0, hipEvent_t e1, hipStream_t s)
{
    uint32_t most = 1;  // tiles of the longest range
    TileRanges r;
    for (int x = 0; x < 9; x++) r.lo[x] = l.lo[x];
    for (int x = 0; x < 8; x++) most = r.lo[x + 1] - r.lo[x] > most ? r.lo[x + 1] - r.lo[x] : most;
    const uint32_t cap = a.grid_cap < 16 ? 1 : a.grid_cap / 16;
    hipExtLaunchKernelGGL((k_rhs<UPWIND, GEN, RK>), dim3(8 * (most < cap ? most : cap)), dim3(512), 0, s, e0, e1, 0, a.in,
                          a.out, a.blocks, a.tile_block, l.order, a.params, a.rk, l.tile0, r);
    return hipGetLastError();
}

template <bool UPWIND, bool RK>
static hipError_t launch_lists(const LaunchArgs &a, hipStream_t s)
{
    const bool fast = a.list[0].lo[8] > a.list[0].lo[0], gen = a.list[1].lo[8] > a.list[1].lo[0];
    hipError_t e = hipSuccess;
    if (fast) e = launch_list<UPWIND, false, RK>(a, a.list[0], a.ev[0], gen ? nullptr : a.ev[1], s);
    if (e == hipSuccess && gen) e = launch_list<UPWIND, true, RK>(a, a.list[1], fast ? nullptr : a.ev[0], a.ev[1], s);
    for (int q = 2; q < 4; q++)
        if (e == hipSuccess && a.ev[q]) e = hipEventRecord(a.ev[q], s);
    return e;
}

hipError_t launch_one_pass(const LaunchArgs &a, hipStream_t s)
{
    if (a.rk.stage >= 0) return a.upwind ? launch_lists<true, true>(a, s) : launch_lists<false, true>(a, s);
    return a.upwind ? launch_lists<true, false>(a, s) : launch_lists<false, false>(a, s);
}

}  // namespace sgr
