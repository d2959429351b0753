// What the RHS kernels share: tile coordinates, index division, the Sommerfeld
// value, eta, and one field's stencils along one axis.
#pragma once

#include "bssn_kernels.h"
#include "stencils.h"

namespace sgr {

struct TileCoord {
    int lt;           // tile id within the block
    int i0, j0, k0;   // padded coordinate of the tile's first interior point
    int oi, oj, ok;   // first coordinate the tile owns along each axis
};

// Tile `lt` of a block tiled with tiles of extents td[] (nt[] tiles per axis).
// The last tile along an axis is shifted back to end at the interior's end,
// so it overlaps its neighbour.  Every tile evaluates derivatives at all its
// points (each tile has its own workspace), but an output point belongs to
// exactly one tile: the one whose unshifted range [GW + td t, GW + td (t + 1))
// holds it.  Stores skip the points a shifted tile shares with the previous
// one, so read-modify-write outputs (the RK4 accumulator) are updated once.
__device__ __forceinline__ TileCoord tile_at(const BlockDesc &B, int lt, const int32_t nt[3], int d0, int d1, int d2)
{
    TileCoord c;
    c.lt = lt;
    const int tx = lt % nt[0];
    const int ty = (lt / nt[0]) % nt[1];
    const int tz = lt / (nt[0] * nt[1]);
    auto origin = [](int tt, int n, int td) {
        const int o = GW + td * tt, last = n - GW - td;
        return o < last ? o : (last > GW ? last : GW);
    };
    c.i0 = origin(tx, B.n[0], d0);
    c.j0 = origin(ty, B.n[1], d1);
    c.k0 = origin(tz, B.n[2], d2);
    c.oi = GW + d0 * tx;
    c.oj = GW + d1 * ty;
    c.ok = GW + d2 * tz;
    return c;
}

// RHS tiling (the block's tile shape) and the constraint pass's 8^3 tiling.
__device__ __forceinline__ TileCoord tile_coord(const BlockDesc &B, uint32_t tile)
{
    return tile_at(B, (int)(tile - B.tile_base), B.ntile, B.tdim[0], B.tdim[1], B.tdim[2]);
}
__device__ __forceinline__ TileCoord tile_coord8(const BlockDesc &B, uint32_t tile)
{
    return tile_at(B, (int)(tile - B.tile_base8), B.ntile8, T, T, T);
}

// Division of a non-negative n < 2^16 by a run-time divisor 2 <= d <= 256
// through its multiplicative inverse m = ceil(2^32 / d): floor(n / d) =
// mulhi(n, m) exactly, since n (m d - 2^32) < n d < 2^32 / d.
struct Div {
    uint32_t m;
};
__device__ __forceinline__ Div make_div(int d) { return Div{0xFFFFFFFFu / (uint32_t)d + 1u}; }
__device__ __forceinline__ int div_q(int n, const Div &v) { return (int)__umulhi((uint32_t)n, v.m); }

// Sommerfeld outgoing-radiation value of one field at a face point
// (bssn/src/rhs.cpp:833-977), evaluated in the reference's order.
__device__ __forceinline__ double sommerfeld(double x, double y, double z, double inv_r, double gx, double gy,
                                             double gz, double fval, double falloff, double asym)
{
    SGR_EXACT
    return -inv_r * (x * gx + y * gy + z * gz + falloff * (fval - asym));
}

__device__ __forceinline__ double coord(double pmin, int i, double h)
{
    SGR_EXACT
    return pmin + i * h;
}

__device__ __forceinline__ double radius(double x, double y, double z)
{
    SGR_EXACT
    return sqrt(x * x + y * y + z * z);
}

__device__ __forceinline__ double ko_add(double v, double sigma, double k)
{
    SGR_EXACT
    return v + sigma * k;
}

// Classic RK4 stage update of one field at one point (see RkArgs).
__device__ __forceinline__ void rk_store(const RkArgs &rk, int f, uint64_t pp, double k)
{
    SGR_EXACT
    const double wk = rk.w * k;
    if (rk.stage == 3) {
        out_put(&rk.next.p[f][pp], rk.acc.p[f][pp] + wk);
        return;
    }
    const double u0 = rk.u0.p[f][pp];
    out_put(&rk.acc.p[f][pp], (rk.stage == 0 ? u0 : rk.acc.p[f][pp]) + wk);
    out_put(&rk.next.p[f][pp], u0 + rk.cn * k);
}

// eta of the Gamma-driver at one point (bssn/src/rhs.cpp:206-219): the
// constant ETA_CONST, damped by (ETA_R0 / r)^ETA_DAMPING_EXP beyond ETA_R0;
// or, under eta_func (GR/bssn.py:52), BSSN_ETA_R0 sqrt(igt^ij d_i chi d_j chi)
// / (1 - chi^p0)^p1 from the point's gt, d chi and chi.
__device__ __forceinline__ double eta_const_at(const Params &P, double x, double y, double z)
{
    double e = P.eta_const;
    const double r = radius(x, y, z);
    if (r >= P.eta_r0) e *= pow(P.eta_r0 / r, P.eta_damping_exp);
    return e;
}
__device__ __forceinline__ double eta_func_at(const Params &P, const double g[6], const double dchi[3], double chi)
{
    double ig[6], h[6];
    inverse_metric(g, ig);
    h[0] = dchi[0] * dchi[0];
    h[1] = dchi[0] * dchi[1];
    h[2] = dchi[0] * dchi[2];
    h[3] = dchi[1] * dchi[1];
    h[4] = dchi[1] * dchi[2];
    h[5] = dchi[2] * dchi[2];
    return P.eta_func_r0 * sqrt(metric_contract(ig, h)) * pow(1.0 - pow(chi, P.eta_power[0]), -P.eta_power[1]);
}

__device__ __forceinline__ double tail_add(double v, double tail)
{
    SGR_EXACT
    return v + tail;
}

// First, advective, Kreiss-Oliger and (want2) pure second derivative of one
// field along one axis at one point.  A tile that reaches a flagged face on
// this axis (lo / hi, uniform over the tile) takes the closure forms: FLAT, the
// ones without divergence (face_taps; k_rhs), else the per-point branches from
// LDS (k_stencil: at its 128 registers the flat forms spill, and the pass takes
// 10.4 instead of 6.4 ms on 512 x 32^3).  Every other tile loads the 7 taps u[-3..3] once into
// registers and evaluates the interior forms from them (same expressions,
// same order: bit-equal to the LDS forms).
template <bool UPWIND, bool FLAT = false>
__device__ __forceinline__ void axis_stencils(const double *c, int s, int pos, int n, bool lo, bool hi, double beta,
                                              const AxisConst &a, bool want2, double &g, double &q, double &k,
                                              double &h)
{
    if (!FLAT && (lo || hi)) {
        g = d1(c, s, pos, n, lo, hi, a);
        q = UPWIND ? adv(c, s, pos, n, lo, hi, beta, a) : g;
        k = ko(c, s, pos, n, lo, hi, a);
        h = want2 ? d2(c, s, pos, n, lo, hi, a) : 0.0;
    } else if (lo || hi) {
        double t[9];
        face_taps(c, s, pos, n, lo, hi, t);
        g = d1_face(t, pos, n, lo, hi, a);
        q = UPWIND ? adv_face(t, pos, n, lo, hi, beta, a) : g;
        k = ko_face(t, pos, n, lo, hi, a);
        h = want2 ? d2_face(t, pos, n, lo, hi, a) : 0.0;
    } else {
        double t[7];
#pragma unroll
        for (int o = 0; o < 7; o++) t[o] = c[(o - 3) * s];
        g = d1_int(t + 3, 1, a);
        q = UPWIND ? ad_int(t + 3, 1, beta > 0.0, a) : g;
        k = ko_int(t + 3, 1, a);
        h = want2 ? d2_int(t + 3, 1, a) : 0.0;
    }
}

}  // namespace sgr
