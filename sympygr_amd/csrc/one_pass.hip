// The BSSN right-hand side in one pass: k_rhs.
//
// The two-pass form stages 69 derivatives and 24 tails of every point in
// memory between the stencils and the algebra.  Here the algebra is folded
// into the field loop instead: fields are processed in an order in which each
// field's derivatives are used up as they appear,
//
//   shift        -> d beta (kept), Gt: lap beta + 1/3 igt d(div beta)
//   gt           -> gt equation; at the last one the connection, the conformal
//                   Ricci terms without d Gt and the Gt terms with CalGt
//   chi          -> chi equation, the chi part of Ricci
//   alpha        -> alpha equation; D_i D_j alpha, the trace-free part, A^ij:
//                   leaves one accumulator per At, Gt and K equation
//   K, Gt, B, At -> each equation is complete when its own field is
//
// so what a point carries from field to field is at most about 50 doubles and
// nothing of it goes to memory.  512 blocks of 32^3 points took 11.9 ms in two
// passes and take 7.4 ms here (10.7 and 6.3 ms without flagged faces).  What bounds it:
// issue of FP64 and LDS instructions by two waves per SIMD that a barrier keeps
// in step.
#include <hip/hip_ext.h>

#include <type_traits>

#include "rhs_common.h"

namespace sgr {

// Keeps the scheduler from mixing the steps of a fold: their intermediate
// values then die before the next step's are formed.
#define SGR_STEP __builtin_amdgcn_sched_barrier(0)

// A value the compiler knows nothing about: keeps it from saving a product
// formed in one step of a fold for the next (held, the saved products of
// igt and C1 alone take a hundred registers; forming them again is one FMA).
__device__ __forceinline__ void renew(double *v, int n)
{
#pragma unroll
    for (int i = 0; i < n; i++) asm volatile("" : "+v"(v[i]));
}

// symmetric slot helpers usable with unrolled loop indices
__host__ __device__ constexpr int sym3(int i, int j) { return i + j + (i > 0 && j > 0 ? 1 : 0); }
__host__ __device__ constexpr int sym_i(int s) { return s < 3 ? 0 : (s < 5 ? 1 : 2); }
__host__ __device__ constexpr int sym_j(int s) { return s < 3 ? s : (s < 5 ? s - 2 : 2); }

// A thread's values parked in LDS lie this far apart (one per thread of the
// workgroup, so a wave's accesses are contiguous).
constexpr int PARK = 512;

// sum_ij a^ij b_ij of two symmetric sets
__device__ __forceinline__ double sym_dot(const double a[6], const double b[6])
{
    return a[0] * b[0] + a[3] * b[3] + a[5] * b[5] + 2.0 * (a[1] * b[1] + a[2] * b[2] + a[4] * b[4]);
}

// Lie derivative terms of a symmetric tensor density of weight -2/3 without
// its advection: t_ik d_j beta^k + t_kj d_i beta^k - 2/3 t_ij div beta
__device__ __forceinline__ double lie_sym(const double t[6], const double *db, double div, int s)
{
    const int i = sym_i(s), j = sym_j(s);
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) v += t[sym3(i, k)] * db[PARK * (3 * k + j)] + t[sym3(k, j)] * db[PARK * (3 * k + i)];
    return v - (2.0 / 3.0) * t[s] * div;
}

// From the 18 first derivatives of the conformal metric, G[3 q + d], to the
// 18 connection coefficients, G[6 k + s] = C2^k_s; adds to R the conformal
// Ricci terms that need neither second derivatives of gt nor d Gt (GR/
// dendro.py:495-499, with the once-raised symbol C1u^l_ab = igt^lm C1_abm), and
// to Gt the terms of CalGt^i = igt^kl C2^i_kl.
__device__ __forceinline__ void fold_connection(double G[18], double R[6], double Gt[3], const double ig[6],
                                                const double *db, double div)
{
    double C1[18];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int i = sym_i(s), j = sym_j(s);
            C1[6 * k + s] = 0.5 * (G[3 * sym3(k, i) + j] + G[3 * sym3(k, j) + i] - G[3 * s + k]);
        }
    SGR_STEP;
    double cal[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int s = 0; s < 6; s++)
            G[6 * k + s] = ig[sym3(k, 0)] * C1[s] + ig[sym3(k, 1)] * C1[6 + s] + ig[sym3(k, 2)] * C1[12 + s];
        cal[k] = sym_dot(ig, &G[6 * k]);
    }
    SGR_STEP;
#pragma unroll
    for (int i = 0; i < 3; i++)
        Gt[i] += (2.0 / 3.0) * cal[i] * div -
                 (cal[0] * db[PARK * 3 * i] + cal[1] * db[PARK * (3 * i + 1)] + cal[2] * db[PARK * (3 * i + 2)]);
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const int i = sym_i(s), j = sym_j(s);
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < 3; k++) v += cal[k] * (C1[6 * i + sym3(j, k)] + C1[6 * j + sym3(i, k)]);
        R[s] += 0.5 * v;
    }
    SGR_STEP;
    renew(C1, 18);
#pragma unroll
    for (int a = 0; a < 3; a++) {
        double cu[9];  // C1u[a][b][l]
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
            for (int l = 0; l < 3; l++)
                cu[3 * b + l] = ig[sym3(l, 0)] * C1[6 * a + sym3(b, 0)] + ig[sym3(l, 1)] * C1[6 * a + sym3(b, 1)] +
                                ig[sym3(l, 2)] * C1[6 * a + sym3(b, 2)];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int l = 0; l < 3; l++) v += G[6 * k + sym3(l, i)] * cu[3 * k + l];
            R[sym3(i, a)] += i == a ? 2.0 * v : v;
        }
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int i = sym_i(s), j = sym_j(s);
            R[s] += G[6 * a + sym3(i, 0)] * cu[3 * j] + G[6 * a + sym3(i, 1)] * cu[3 * j + 1] +
                    G[6 * a + sym3(i, 2)] * cu[3 * j + 2];
        }
        SGR_STEP;
    }
}

// the chi part of Ricci (GR/dendro.py:509-518) from d chi and its second
// derivatives h
__device__ __forceinline__ void fold_chi(double R[6], const double G[18], const double g[6], const double ig[6],
                                         double ichi, const double dc[3], const double h[6])
{
    double dd[6], q[6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        dd[s] = h[s] - (G[s] * dc[0] + G[6 + s] * dc[1] + G[12 + s] * dc[2]);
        q[s] = dd[s] - 1.5 * ichi * (dc[sym_i(s)] * dc[sym_j(s)]);
    }
    const double tr = sym_dot(ig, q);
#pragma unroll
    for (int s = 0; s < 6; s++)
        R[s] += 0.5 * ichi * (dd[s] + g[s] * tr) - 0.25 * (ichi * ichi) * (dc[sym_i(s)] * dc[sym_j(s)]);
}

// Everything that needs D_i D_j alpha or A^ij (GR/bssn.py:67-100): in R the
// Ricci tensor without its d Gt terms, out T the At equation without them,
// Gt completed but for d K, Kr the K equation.
__device__ __forceinline__ void fold_alpha(double T[6], double Gt[3], double &Kr, const double R[6],
                                           const double G[18], const double g[6], const double ig[6],
                                           const double *db, double div, double alpha, double chi, double ichi,
                                           double K, const double dc[3], const double da[3], const double h[6],
                                           const double A[6])
{
    double X[6];
    {
        double up[3];
#pragma unroll
        for (int i = 0; i < 3; i++)
            up[i] = ig[sym3(i, 0)] * dc[0] + ig[sym3(i, 1)] * dc[1] + ig[sym3(i, 2)] * dc[2];
        const double ud = up[0] * da[0] + up[1] * da[1] + up[2] * da[2];
        double dd[6];
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int i = sym_i(s), j = sym_j(s);
            dd[s] = h[s] - (G[s] * da[0] + G[6 + s] * da[1] + G[12 + s] * da[2]) +
                    0.5 * ichi * (da[i] * dc[j] + da[j] * dc[i] - g[s] * ud);
            X[s] = alpha * R[s] - dd[s];
        }
        Kr = -chi * sym_dot(ig, dd);
    }
    SGR_STEP;
    const double tr3 = (1.0 / 3.0) * sym_dot(ig, X);
    double M[9], AU[6];  // igt^ik A_kj and A^ij
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            M[3 * i + j] = ig[sym3(i, 0)] * A[sym3(0, j)] + ig[sym3(i, 1)] * A[sym3(1, j)] + ig[sym3(i, 2)] * A[sym3(2, j)];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const int i = sym_i(s), j = sym_j(s);
        const double aa = A[sym3(i, 0)] * M[j] + A[sym3(i, 1)] * M[3 + j] + A[sym3(i, 2)] * M[6 + j];
        T[s] = lie_sym(A, db, div, s) + chi * (X[s] - g[s] * tr3) + alpha * (K * A[s] - 2.0 * aa);
        AU[s] = M[3 * i] * ig[sym3(0, j)] + M[3 * i + 1] * ig[sym3(1, j)] + M[3 * i + 2] * ig[sym3(2, j)];
    }
    SGR_STEP;
    Kr += alpha * ((1.0 / 3.0) * K * K + sym_dot(A, AU));
    const double a3 = 3.0 * alpha * ichi;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double v = 2.0 * alpha * sym_dot(&G[6 * i], AU);
#pragma unroll
        for (int j = 0; j < 3; j++) v -= AU[sym3(i, j)] * (2.0 * da[j] + a3 * dc[j]);
        Gt[i] += v;
    }
}

// The block table and the tile map are constant while k_rhs runs: read through
// the constant address space they are scalar loads (as plain global memory,
// which the kernel's own stores might alias, they are vector loads).
#define SGR_CONST_MEM __attribute__((address_space(4)))
#define SGR_GLOBAL __attribute__((address_space(1)))
typedef const SGR_CONST_MEM BlockDesc *ConstBlock;
__device__ __forceinline__ AxisConst axis_of(ConstBlock B, int d)
{
    AxisConst a;
    a.h = B->ax[d].h, a.by60 = B->ax[d].by60, a.by12 = B->ax[d].by12, a.sq180 = B->ax[d].sq180, a.sq12 = B->ax[d].sq12;
    a.by2 = B->ax[d].by2, a.ko_pre = B->ax[d].ko_pre, a.smr3 = B->ax[d].smr3, a.smr2 = B->ax[d].smr2, a.smr1 = B->ax[d].smr1;
    return a;
}
// The first words of a block's descriptor, one per lane of a vector register:
// fetched for the next tile while the current one is worked on (a scalar load
// would be waited for with the next LDS access) and read with v_readlane.
struct DescWords {
    int w;
    __device__ __forceinline__ void load(const BlockDesc *B, int lane)
    {
        static_assert(offsetof(BlockDesc, n) == 16 && offsetof(BlockDesc, ntile) == 28 && offsetof(BlockDesc, tdim) == 40 &&
                          offsetof(BlockDesc, bflag) == 64 && offsetof(BlockDesc, tile_base) == 68,
                      "word numbers below");
        w = ((const SGR_GLOBAL int *)(uint64_t)B)[lane < 18 ? lane : 0];
    }
    __device__ __forceinline__ int at(int k) const { return __builtin_amdgcn_readlane(w, k); }
    __device__ __forceinline__ uint64_t offset() const { return (uint64_t)(uint32_t)at(1) << 32 | (uint32_t)at(0); }
    __device__ __forceinline__ int n(int k) const { return at(4 + k); }
    __device__ __forceinline__ int tdim(int k) const { return at(10 + k); }
    __device__ __forceinline__ uint32_t bflag() const { return (uint32_t)at(16); }
    __device__ __forceinline__ TileCoord coord(uint32_t tile) const
    {
        BlockDesc d;
#pragma unroll
        for (int k = 0; k < 3; k++) d.n[k] = n(k);
        const int32_t nt[3] = {at(7), at(8), at(9)};
        return tile_at(d, (int)(tile - (uint32_t)at(17)), nt, tdim(0), tdim(1), tdim(2));
    }
};

// Field order of k_rhs: the 11 fields with second derivatives first.
constexpr int FUSED_D2 = 11;
__host__ __device__ constexpr int fused_field(int p)
{
    return p < 3 ? 6 + p : p < 9 ? 9 + p : p == 9 ? 1 : p == 10 ? 0 : p == 11 ? 2 : p < 15 ? p - 9 : p < 18 ? p - 6 : p;
}

// pow, out of line: inlined, its coefficients are hoisted out of the tile loop
// and their registers spill.
__device__ __attribute__((noinline)) double eta_pow(double x, double y) { return pow(x, y); }

// The arrays of the fields in k_rhs's order, one pointer per lane: fetched with
// v_readlane instead of a scalar load with its wait in every field.
struct FieldTable {
    int lo, hi;
    __device__ __forceinline__ void set(const double *p) { lo = (int)(uint32_t)(uint64_t)p, hi = (int)((uint64_t)p >> 32); }
    __device__ __forceinline__ SGR_GLOBAL double *get(int p) const
    {
        return (SGR_GLOBAL double *)((uint64_t)(uint32_t)__builtin_amdgcn_readlane(lo, p) |
                                     (uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, p) << 32);
    }
};

// The tiles of one k_rhs launch: entries lo[x] .. lo[x + 1] - 1 of its list
// belong to XCD x (workgroups go to the XCDs round-robin by id).
struct TileRanges {
    uint32_t lo[9];
};

// One 512-thread workgroup per CU (2 waves per SIMD, so a point's state fits
// in 256 registers; LDS 148 KB), one point per thread, one tile at a time.
//   U   the halo tile of a field, two buffers: while one is read, the next
//       field's tile arrives (loads issued a whole field ahead) and is stored
//       into the other
//   DX  D_x u and DY D_y u for the mixed derivatives, two buffers each
//   DB  the thread's first derivatives of the shift, parked
// With both double-buffered a field takes one barrier: stencils and the stores
// of DX, DY and the next U before it, mixed derivatives and algebra after it.
// The general shapes have room for one DX and DY and take a second barrier.
// The grid is persistent: a workgroup takes every (gridDim.x / 8)-th tile of
// its XCD's range, and the next tile's first fields and point values are
// fetched during the last fields of the current one.  Tiles that reach a
// flagged face run their own copy of the code, the only one with the closure
// forms; `order` lists each range's other tiles first, so that a CU works in
// one copy at a time (both do not fit its instruction cache).
// order: tile numbers relative to tile0, or null for 0, 1, 2, ...
// RK: an RK stage's update instead of the plain RHS (rk.stage >= 0).
template <bool UPWIND, bool GEN, bool RK>
__global__ __launch_bounds__(512, 2) void k_rhs(FieldPtrs in, OutPtrs out, const BlockDesc *__restrict__ blocks,
                                                const uint32_t *__restrict__ tile_block,
                                                const uint32_t *__restrict__ order, Params P, RkArgs rk,
                                                uint32_t tile0, TileRanges ranges)
{
    constexpr int NT = 512;
    constexpr int RS8 = 24, PS8 = RS8 * TH;       // 8^3: padded halo rows (conflict-free, see k_stencil)
    constexpr int USZ = GEN ? GEN_U_CAP : PS8 * TH;
    constexpr int DXSZ = GEN ? GEN_DX_CAP : T * TH * TH, DYSZ = GEN ? GEN_DY_CAP : T * T * TH;
    constexpr int NPF = GEN ? 4 : 3;              // halo loads per thread, 16 bytes each
    constexpr int NB2 = GEN ? 1 : 2;              // buffers of DX and DY
    __shared__ __align__(16) double U[2 * USZ];
    __shared__ double DX[NB2 * DXSZ];
    __shared__ double DY[NB2 * DYSZ];
    __shared__ double DB[9 * NT];                 // each thread's d_j beta^i, at 3 i + j
    __shared__ double SP[3];                      // sigma, lambda_2, 1 - lambda_3

    const int t = threadIdx.x;
    const uint32_t stride = gridDim.x >> 3, end = ranges.lo[(blockIdx.x & 7) + 1];
    uint32_t m = ranges.lo[blockIdx.x & 7] + (blockIdx.x >> 3);  // place in the list
    if (m >= end) return;
    // the thread index, opaque to the compiler: what derives from it is
    // recomputed where it is needed instead of held (and spilled: a reload waits
    // for every load issued before it, the next halo tile's too)
    auto thread = []() __attribute__((always_inline)) {
        int v = threadIdx.x;
        asm volatile("" : "+v"(v));
        return v;
    };
    // vector loads of one word (lane-dependent address, so that they stay such)
    auto tile_of = [&](uint32_t m) __attribute__((always_inline)) -> uint32_t {
        return order ? ((const SGR_GLOBAL uint32_t *)(uint64_t)order)[m + (thread() >> 10)] : m;
    };
    auto block_of = [&](uint32_t tile) __attribute__((always_inline)) -> uint32_t {
        return ((const SGR_GLOBAL uint32_t *)(uint64_t)tile_block)[tile + (thread() >> 10)];
    };
    auto first = [](uint32_t v) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };

    FieldTable tin, tout, tnext, tu0;  // RK: tout the accumulator
    {
        const int l = t & 63, f = l < NF ? fused_field(l) : 0;
        tin.set(in.p[f]);
        if (RK) {
            tout.set(rk.acc.p[f]);
            tnext.set(rk.next.p[f]);
            tu0.set(rk.u0.p[f]);
        } else {
            tout.set(out.p[f]);
        }
    }
    // (read from LDS where they are used: scalar loads of them were waited for
    // in every field, registers for them spilled)
    if (t == 0) SP[0] = P.ko_sigma, SP[1] = P.lambda[2], SP[2] = 1.0 - P.lambda[3];

    // What the halo loads of one tile need.  A load takes two neighbours of a
    // row (16 bytes, 8-byte aligned), half as many instructions for the same
    // bytes as single values.  8^3: thread t < 490 holds pair t % 98 of the 14 x
    // 14 plane, planes t / 98 + 5 q.  General: pairs t + 512 q of the halo, the
    // last one of an odd row shifted back to end with it.
    typedef double Pair __attribute__((ext_vector_type(2), aligned(8)));
    constexpr int PP = TH * TH / 2;
    uint64_t lbase = 0;             // uniform: halo corner in the field arrays
    int ln0 = 0, ln01 = 0;          // 8^3: the block's y and z strides
    int src[GEN ? NPF : 1], dst[GEN ? NPF : 1];
    const bool loader = GEN || t < 5 * PP;
    Pair pf[NPF];
    auto aim = [&](const DescWords &D, const TileCoord &tc) __attribute__((always_inline)) {
        const int t = thread();
        const int n0 = D.n(0), n01 = n0 * D.n(1);
        lbase = D.offset() + (tc.i0 - GW) + (uint64_t)n0 * (tc.j0 - GW) + (uint64_t)n01 * (tc.k0 - GW);
        if constexpr (GEN) {
            const int HX = D.tdim(0) + 2 * GW, HY = D.tdim(1) + 2 * GW, PX = (HX + 1) >> 1;
            const int np = PX * HY * (D.tdim(2) + 2 * GW);
            const Div dPX = make_div(PX), dHY = make_div(HY);
#pragma unroll
            for (int q = 0; q < NPF; q++) {
                const int e = t + NT * q, r = div_q(e, dPX), ez = div_q(r, dHY), ex = min(2 * (e - r * PX), HX - 2);
                src[q] = e < np ? ex + n0 * (r - ez * HY) + n01 * ez : 0;
                dst[q] = e < np ? ex + HX * r : -1;
            }
        } else {
            ln0 = n0, ln01 = n01;
        }
    };
    auto fetch = [&](int p) __attribute__((always_inline)) {
        const SGR_GLOBAL double *s = tin.get(p) + lbase;
        if constexpr (GEN) {
#pragma unroll
            for (int q = 0; q < NPF; q++) pf[q] = *(const SGR_GLOBAL Pair *)(s + src[q]);
        } else if (loader) {
            const int t = thread();
            const int pz = t / PP, py = (t - pz * PP) / (TH / 2), px = 2 * (t - pz * PP - py * (TH / 2));
            const int e = px + ln0 * py + ln01 * pz;
            pf[0] = *(const SGR_GLOBAL Pair *)(s + e);
            pf[1] = *(const SGR_GLOBAL Pair *)(s + (e + 5 * ln01));
            pf[2] = *(const SGR_GLOBAL Pair *)(s + (pz < 4 ? e + 10 * ln01 : e));  // planes 10 .. 13
        }
    };
    int pdst[GEN ? NPF : 1];  // where `pf` goes
    auto put = [&](double *u) __attribute__((always_inline)) {
        const int t = thread();
        const int pz = t / PP, py = (t - pz * PP) / (TH / 2), px = 2 * (t - pz * PP - py * (TH / 2));
        const int d8 = px + RS8 * py + PS8 * pz;
        if (loader) {
#pragma unroll
            for (int q = 0; q < NPF; q++) {
                if (GEN) {
                    if (pdst[q] >= 0) *(Pair *)(u + pdst[q]) = pf[q];
                } else if (q < 2 || pz < 4) {
                    *(double2 *)(u + d8 + 5 * PS8 * q) = double2{pf[q].x, pf[q].y};
                }
            }
        }
    };

    double pv[10];  // the point's shift, conformal metric and lapse, of the tile `aim` points at
    auto point_of = [&](int t, const DescWords &D, int &lx, int &ly, int &lz, bool &has) __attribute__((always_inline)) {
        if (GEN) {
            const int TX = D.tdim(0), TY = D.tdim(1), np = TX * TY * D.tdim(2);
            has = t < np;
            const int tt = has ? t : np - 1;  // spare threads repeat the last point and store nothing
            const int r = div_q(tt, make_div(TX));
            lz = div_q(r, make_div(TY));
            lx = tt - r * TX;
            ly = r - lz * TY;
        } else {
            has = true;
            lx = t & 7, ly = (t >> 3) & 7, lz = t >> 6;
        }
    };
    auto fetch_point = [&](const DescWords &D) __attribute__((always_inline)) {
        int lx, ly, lz;
        bool has;
        point_of(thread(), D, lx, ly, lz, has);
        const int o = (lx + GW) + D.n(0) * ((ly + GW) + D.n(1) * (lz + GW));
#pragma unroll
        for (int q = 0; q < 10; q++) pv[q] = (tin.get(q < 9 ? q : 10) + lbase)[o];
    };
    auto keep_dst = [&]() __attribute__((always_inline)) {
        if constexpr (GEN) {
#pragma unroll
            for (int q = 0; q < NPF; q++) pdst[q] = dst[q];
        }
    };

    int b = 0;  // the buffers in use

    // One tile: its descriptor words D and block nb; the next one's place in the
    // list, and, filled on the way, its tile, block and descriptor words.
    auto run_tile = [&](auto face_, const DescWords &D, const TileCoord &tc, const ConstBlock B, uint32_t mnext,
                        uint32_t &next, uint32_t &nnext, DescWords &Dnext, TileCoord &tnc) __attribute__((always_inline)) {
        constexpr bool FACE = decltype(face_)::value;
        const int TX = GEN ? D.tdim(0) : T, TY = GEN ? D.tdim(1) : T, TZ = GEN ? D.tdim(2) : T;
        const int HX = TX + 2 * GW, HY = TY + 2 * GW;
        const int RS = GEN ? HX : RS8, PS = GEN ? HX * HY : PS8;
        const int DXZ = TX * HY, DYZ = TX * TY;
        const int n0 = D.n(0), n1 = D.n(1), n2 = D.n(2);
        const uint32_t bflag = D.bflag();
        const bool lo0 = FACE && (bflag & 1u), hi0 = FACE && (bflag & 2u), lo1 = FACE && (bflag & 4u);
        const bool hi1 = FACE && (bflag & 8u), lo2 = FACE && (bflag & 16u), hi2 = FACE && (bflag & 32u);
        // closure forms: tiles within three points of the face (uniform)
        const bool clo0 = lo0 && tc.i0 < GW + 3, chi0 = hi0 && tc.i0 + TX - 1 >= n0 - GW - 3;
        const bool clo1 = lo1 && tc.j0 < GW + 3, chi1 = hi1 && tc.j0 + TY - 1 >= n1 - GW - 3;
        const bool clo2 = lo2 && tc.k0 < GW + 3, chi2 = hi2 && tc.k0 + TZ - 1 >= n2 - GW - 3;
        const uint64_t obase = D.offset();

        bool own;  // is the point this tile's (tile_at)?
        int gp;    // its place in the block
        {
            int lx, ly, lz;
            bool has;
            point_of(thread(), D, lx, ly, lz, has);
            const int pi = tc.i0 + lx, pj = tc.j0 + ly, pk = tc.k0 + lz;
            own = has && pi >= tc.oi && pj >= tc.oj && pk >= tc.ok;
            gp = pi + n0 * (pj + n1 * pk);
        }
        double bv[3], g[6], ig[6];
#pragma unroll
        for (int d = 0; d < 3; d++) bv[d] = pv[d];
#pragma unroll
        for (int q = 0; q < 6; q++) g[q] = pv[3 + q];
        const double alpha = pv[9];
        inverse_metric(g, ig);
        double G[18], R[6], Gt[3], gdb[3], dc[3], div = 0.0, Kv = 0.0, Kr = 0.0, chi = 1.0, eta = 0.0, es = 0.0;

        // Fields 0 .. p of a tile, one at a time: `begin` evaluates field p's
        // stencils (and moves the pipeline of halo tiles on), `finish` stores
        // its equation, alg + (lin + sigma KO).
        struct FieldVals {
            double g[3], h[6];           // first and second derivatives
            double adv, ko, bc, uv, ex;  // bc: the whole output of a flagged-face point
            double u0v, acv;             // RK stage inputs
            SGR_GLOBAL double *out, *next;  // where the equation goes (RK stage: accumulator and next stage)
            bool face;
        };
        double A[6];  // At at the point, from field 10 on
        auto begin = [&](auto d2_, auto last_, int p, FieldVals &v) __attribute__((always_inline)) {
            constexpr bool D2 = decltype(d2_)::value;
            const int f = fused_field(p);
            const int t = thread();
            int lx, ly, lz;
            bool has;
            point_of(t, D, lx, ly, lz, has);
            const int pi = tc.i0 + lx, pj = tc.j0 + ly, pk = tc.k0 + lz;
            v.out = tout.get(p) + obase;
            if (RK) v.next = tnext.get(p) + obase;
            v.face = FACE && ((lo0 && pi == GW) || (hi0 && pi == n0 - GW - 1) || (lo1 && pj == GW) ||
                                   (hi1 && pj == n1 - GW - 1) || (lo2 && pk == GW) || (hi2 && pk == n2 - GW - 1));
            const int uc = (lx + GW) + RS * (ly + GW) + PS * (lz + GW);
            const int cx = lx + TX * (ly + GW) + DXZ * (lz + GW), cy = lx + TX * ly + DYZ * (lz + GW);
            const double *c = &U[b * USZ + uc];
            double *dx = &DX[(NB2 - 1) * b * DXSZ], *dy = &DY[(NB2 - 1) * b * DYSZ];
            // the block's constants, read again in every field: fewer scalar
            // registers held across it
            uint64_t bp = (uint64_t)B;
            asm volatile("" : "+s"(bp));
            const AxisConst a0 = axis_of((ConstBlock)bp, 0), a1 = axis_of((ConstBlock)bp, 1), a2 = axis_of((ConstBlock)bp, 2);
            // point values this field's algebra needs, and the RK stage's
            v.u0v = v.acv = v.ex = 0.0;
            if (RK) {
                if (rk.stage < 3) v.u0v = (tu0.get(p) + obase)[gp];
                if (rk.stage > 0) v.acv = v.out[gp];
            }
            if (D2) v.ex = (tin.get(p < 9 ? 15 + p : 11) + obase)[gp];  // B^k, At_q; K
            double &g0 = v.g[0], &g1 = v.g[1], &g2 = v.g[2], q0, q1, q2, k0, k1, k2, *h = v.h;
            axis_stencils<UPWIND, true>(c, 1, pi, n0, clo0, chi0, bv[0], a0, D2, g0, q0, k0, h[0]);
            axis_stencils<UPWIND, true>(c, RS, pj, n1, clo1, chi1, bv[1], a1, D2, g1, q1, k1, h[3]);
            axis_stencils<UPWIND, true>(c, PS, pk, n2, clo2, chi2, bv[2], a2, D2, g2, q2, k2, h[5]);
            v.uv = c[0];
            if (D2) {
                if (p == 10) {
#pragma unroll
                    for (int q = 0; q < 6; q++) A[q] = (tin.get(18 + q) + obase)[gp];
                }
                dx[cx] = g0;
                dy[cy] = g1;
                const double *u = &U[b * USZ];
                // D_x and D_y on the tile's z halo planes, D_x on the y halo
                // rows of its z planes (the corners are never read)
                if constexpr (GEN) {
                    const int NB = TX * TY * (2 * GW), NA = TX * (2 * GW) * TZ;
                    const Div dTX = make_div(TX), dTY = make_div(TY);
                    for (int e = t; e < NA + NB; e += NT) {
                        if (e < NB) {
                            const int r = div_q(e, dTX), rz = div_q(r, dTY);
                            const int xx = e - r * TX, yy = r - rz * TY, zz = rz < GW ? rz : rz + TZ;
                            const double *cu = u + (xx + GW) + RS * (yy + GW) + PS * zz;
                            dx[xx + TX * (yy + GW) + DXZ * zz] = d1_tile(cu, 1, tc.i0 + xx, n0, clo0, chi0, a0);
                            dy[xx + TX * yy + DYZ * zz] = d1_tile(cu, RS, tc.j0 + yy, n1, clo1, chi1, a1);
                        } else {
                            const int r0 = e - NB, r = div_q(r0, dTX), zt = r / (2 * GW), ry = r - zt * (2 * GW);
                            const int xx = r0 - r * TX, yy = ry < GW ? ry : ry + TY, zz = GW + zt;
                            dx[xx + TX * yy + DXZ * zz] =
                                d1_tile(u + (xx + GW) + RS * yy + PS * zz, 1, tc.i0 + xx, n0, clo0, chi0, a0);
                        }
                    }
                } else {
                    // 18 planes or rows of 64 cells: D_x and D_y of the six z halo
                    // planes, D_x of the six y halo rows.  Two to every wave, and the
                    // last two rows to all, 16 cells each.
                    const int w = __builtin_amdgcn_readfirstlane(t >> 6), xx = t & 7, m8 = (t >> 3) & 7;
                    auto z_plane = [&](int p6, int yy, bool is_y) __attribute__((always_inline)) {
                        const int zz = p6 < GW ? p6 : p6 + T;
                        const double *cu = u + (xx + GW) + RS * (yy + GW) + PS * zz;
                        if (is_y) dy[xx + T * yy + DYZ * zz] = d1_tile(cu, RS, tc.j0 + yy, n1, clo1, chi1, a1);
                        else dx[xx + T * (yy + GW) + DXZ * zz] = d1_tile(cu, 1, tc.i0 + xx, n0, clo0, chi0, a0);
                    };
                    auto y_row = [&](int ry, int zz) __attribute__((always_inline)) {
                        const int yy = ry < GW ? ry : ry + T;
                        dx[xx + T * yy + DXZ * zz] =
                            d1_tile(u + (xx + GW) + RS * yy + PS * zz, 1, tc.i0 + xx, n0, clo0, chi0, a0);
                    };
                    if (w < 6) {
                        z_plane(w, m8, false);
                        z_plane(w, m8, true);
                    } else {
                        y_row(w - 6, m8 + GW);
                        y_row(w - 4, m8 + GW);
                    }
                    if ((t & 63) < 16) y_row(4 + (m8 & 1), w + GW);
                }
            }
            put(&U[(1 - b) * USZ]);  // the next field's halo tile
            __syncthreads();
            // (what was loaded for this field is waited for here: behind the next
            // loads it would have to wait for them too)
            asm volatile("" : "+v"(v.ex), "+v"(v.u0v), "+v"(v.acv));
            if (D2 && p == 10) renew(A, 6);
            // the loads of the field after it (at the end, of the next tile's first;
            // its second: at its start)
            if constexpr (!decltype(last_)::value) {
                keep_dst();
                fetch(p + 2 < NF ? p + 2 : 0);
            }

            // the terms linear in the field's own advective and KO stencils
            {
                SGR_EXACT
                v.adv = (bv[0] * q0 + bv[1] * q1) + bv[2] * q2;
                v.ko = (k0 + k1) + k2;
            }
            v.bc = 0.0;
            if (v.face) {  // the Sommerfeld value replaces the right-hand side, then + sigma KO
                const double x = coord(B->pmin[0], pi, a0.h), y = coord(B->pmin[1], pj, a1.h);
                const double z = coord(B->pmin[2], pk, a2.h);
                v.bc = ko_add(sommerfeld(x, y, z, 1.0 / radius(x, y, z), g0, g1, g2, v.uv, bc_falloff(f), bc_asym(f)),
                              SP[0], v.ko);
            }
            if constexpr (D2) {
                const double *cxp = &dx[cx], *cyp = &dy[cy];
                h[1] = d1_tile(cxp, TX, pj, n1, clo1, chi1, a1);   // D_y D_x
                h[2] = d1_tile(cxp, DXZ, pk, n2, clo2, chi2, a2);  // D_z D_x
                h[4] = d1_tile(cyp, DYZ, pk, n2, clo2, chi2, a2);  // D_z D_y
                if (NB2 == 1) __syncthreads();  // DX and DY are read
            }
            b ^= 1;
        };
        auto finish = [&](const FieldVals &v, double alg, double lin) __attribute__((always_inline)) {
            SGR_EXACT
            if (!own) return;
            const double k = v.face ? v.bc : alg + (lin + SP[0] * v.ko);
            if (!RK) {
                v.out[gp] = k;
                return;
            }
            const double wk = rk.w * k;
            if (rk.stage == 3) {
                v.next[gp] = v.acv + wk;
                return;
            }
            v.out[gp] = (rk.stage == 0 ? v.u0v : v.acv) + wk;
            v.next[gp] = v.u0v + rk.cn * k;
        };
        auto times = [](double a, double b) __attribute__((always_inline)) {
            SGR_EXACT
            return a * b;
        };
        double *const db = &DB[t];
        auto shift = [&](auto k_, const FieldVals &v) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                db[PARK * (3 * k + j)] = v.g[j];
                gdb[j] = k == 0 ? v.h[sym3(k, j)] : gdb[j] + v.h[sym3(k, j)];
            }
            div = k == 0 ? v.g[k] : div + v.g[k];
            Gt[k] = metric_contract(ig, v.h);
            if (k == 2) {
#pragma unroll
                for (int i = 0; i < 3; i++)
                    Gt[i] += (1.0 / 3.0) * (ig[sym3(i, 0)] * gdb[0] + ig[sym3(i, 1)] * gdb[1] + ig[sym3(i, 2)] * gdb[2]);
            }
            finish(v, 0.75 * (P.lambda_f[0] + P.lambda_f[1] * alpha) * v.ex, times(P.lambda[1], v.adv));
        };
        auto metric = [&](auto q_, const FieldVals &v) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
#pragma unroll
            for (int j = 0; j < 3; j++) G[3 * q + j] = v.g[j];
            R[q] = -0.5 * metric_contract(ig, v.h);
            return lie_sym(g, db, div, q) - 2.0 * alpha * v.ex;
        };
        auto gamma = [&](auto k_, const FieldVals &v) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value;
            const double ac = alpha * chi;
#pragma unroll
            for (int s = 0; s < 6; s++) {
                const int i = sym_i(s), j = sym_j(s);
                R[s] += ac * (0.5 * (g[sym3(k, i)] * v.g[j] + g[sym3(k, j)] * v.g[i]) - (1.0 / 3.0) * g[s] * v.g[k]);
            }
            const double alg = Gt[k];
            Gt[k] += SP[2] * v.adv;  // what B^k's equation takes of this one
            return alg;
        };

#define SGR_K(n) std::integral_constant<int, n>{}
        uint32_t word = tile_of(mnext);
#pragma unroll 1
        for (int p = 0; p < 3; p++) {  // the shift
            FieldVals v;
            begin(std::true_type{}, std::false_type{}, p, v);
            if (p == 0) shift(SGR_K(0), v);
            else if (p == 1) shift(SGR_K(1), v);
            else shift(SGR_K(2), v);
        }
        next = first(word);
        word = block_of(next);
#pragma unroll 1
        for (int p = 3; p < 9; p++) {  // gt
            FieldVals v;
            begin(std::true_type{}, std::false_type{}, p, v);
            double alg;
            switch (p) {
            case 3: alg = metric(SGR_K(0), v); break;
            case 4: alg = metric(SGR_K(1), v); break;
            case 5: alg = metric(SGR_K(2), v); break;
            case 6: alg = metric(SGR_K(3), v); break;
            case 7: alg = metric(SGR_K(4), v); break;
            default: alg = metric(SGR_K(5), v); break;
            }
            finish(v, alg, v.adv);
        }
        nnext = first(word);
        fold_connection(G, R, Gt, ig, db, div);
        {
            FieldVals v;
#pragma unroll 1
            for (int p = 9; p < 11; p++) {  // chi, alpha
                begin(std::true_type{}, std::false_type{}, p, v);
                if (p == 9) {
                    chi = v.uv;
                    Kv = v.ex;
#pragma unroll
                    for (int d = 0; d < 3; d++) dc[d] = v.g[d];
                    fold_chi(R, G, g, ig, 1.0 / chi, dc, v.h);
                    if (P.eta_func) {
                        const double dd[6] = {dc[0] * dc[0], dc[0] * dc[1], dc[0] * dc[2],
                                              dc[1] * dc[1], dc[1] * dc[2], dc[2] * dc[2]};
                        es = metric_contract(ig, dd);
                    }
                }
                finish(v, p == 9 ? (2.0 / 3.0) * chi * (alpha * Kv - div) : -2.0 * alpha * Kv,
                       p == 9 ? v.adv : times(P.lambda[0], v.adv));
            }
            double Tq[6];
            fold_alpha(Tq, Gt, Kr, R, G, g, ig, db, div, alpha, chi, 1.0 / chi, Kv, dc, v.g, v.h, A);
#pragma unroll
            for (int q = 0; q < 6; q++) R[q] = Tq[q];  // from here on the At accumulators
        }
        Dnext.load(blocks + nnext, thread() & 63);
#pragma unroll 1
        for (int p = FUSED_D2; p < 15; p++) {  // K, Gt
            FieldVals v;
            begin(std::false_type{}, std::false_type{}, p, v);
            double alg;
            switch (p) {
            case 11:
#pragma unroll
                for (int i = 0; i < 3; i++)
                    Gt[i] -= (4.0 / 3.0) * alpha * (ig[sym3(i, 0)] * v.g[0] + ig[sym3(i, 1)] * v.g[1] + ig[sym3(i, 2)] * v.g[2]);
                alg = Kr;
                break;
            case 12: alg = gamma(SGR_K(0), v); break;
            case 13: alg = gamma(SGR_K(1), v); break;
            default: alg = gamma(SGR_K(2), v); break;
            }
            finish(v, alg, v.adv);
        }
        if (P.eta_func) {
            eta = P.eta_func_r0 * sqrt(es) * eta_pow(1.0 - eta_pow(chi, P.eta_power[0]), -P.eta_power[1]);
        } else {
            int lx, ly, lz;
            bool has;
            point_of(thread(), D, lx, ly, lz, has);
            const double r = radius(coord(B->pmin[0], tc.i0 + lx, B->ax[0].h), coord(B->pmin[1], tc.j0 + ly, B->ax[1].h),
                                    coord(B->pmin[2], tc.k0 + lz, B->ax[2].h));
            eta = P.eta_const;
            if (r >= P.eta_r0) eta *= eta_pow(P.eta_r0 / r, P.eta_damping_exp);
        }
#pragma unroll 1
        for (int p = 15; p < NF - 2; p++) {  // B, At
            FieldVals v;
            begin(std::false_type{}, std::false_type{}, p, v);
            double alg;
            switch (p) {
            case 15: alg = Gt[0] - eta * v.uv; break;
            case 16: alg = Gt[1] - eta * v.uv; break;
            case 17: alg = Gt[2] - eta * v.uv; break;
            case 18: alg = R[0]; break;
            case 19: alg = R[1]; break;
            case 20: alg = R[2]; break;
            default: alg = R[3]; break;
            }
            finish(v, alg, p < 18 ? times(SP[1], v.adv) : v.adv);
        }
        // the last but one fetches for the next tile (the last tile: its own again, unused)
        tnc = Dnext.coord(next);
        aim(Dnext, tnc);
        fetch_point(Dnext);
        {
            FieldVals v;
            begin(std::false_type{}, std::false_type{}, NF - 2, v);
            finish(v, R[4], v.adv);
        }
        {
            FieldVals v;
            begin(std::false_type{}, std::true_type{}, NF - 1, v);
            finish(v, R[5], v.adv);
        }
#undef SGR_K
    };

    uint32_t tile = first(tile_of(m)), nb = first(block_of(tile));
    DescWords D;
    D.load(blocks + nb, t & 63);
    TileCoord tc = D.coord(tile);
    aim(D, tc);
    fetch(0);
    fetch_point(D);
    keep_dst();
    put(U);
    __syncthreads();
    for (;;) {
        keep_dst();
        fetch(1);
        m += stride;
        const uint32_t mnext = m < end ? m : m - stride;  // (the last tile's own again, unused)
        bool face = false;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int o = d == 0 ? tc.i0 : d == 1 ? tc.j0 : tc.k0;
            face |= ((D.bflag() >> (2 * d)) & 1u && o < GW + 3) ||
                    ((D.bflag() >> (2 * d + 1)) & 1u && o + (GEN ? D.tdim(d) : T) - 1 >= D.n(d) - GW - 3);
        }
        uint32_t next = 0, nnext = 0;
        DescWords Dnext;
        TileCoord tnc;
        const ConstBlock B = (ConstBlock)(uint64_t)(blocks + nb);
        if (face) run_tile(std::true_type{}, D, tc, B, mnext, next, nnext, Dnext, tnc);
        else run_tile(std::false_type{}, D, tc, B, mnext, next, nnext, Dnext, tnc);
        if (m >= end) break;
        tile = next, nb = nnext, D = Dnext, tc = tnc;
    }
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
