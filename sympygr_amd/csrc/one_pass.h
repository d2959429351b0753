// The right-hand side in one pass (k_rhs, one_pass.hip), and on the same path
// the constraints and Psi4 (k_monitor, monitor.hip).
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
// passes and take 7.3 ms here (10.7 and 6.3 ms without flagged faces).  What bounds it:
// issue of FP64 and LDS instructions by two waves per SIMD that a barrier keeps
// in step.
#pragma once

#include <hip/hip_ext.h>

#include <type_traits>

#include "rhs_common.h"

namespace sgr {

// Products fused into sums where the source says so, statement by statement (the
// compiler's own choice differs between the kernels of the two tile shapes, whose
// results have to be the same bits).
#pragma clang fp contract(on)

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
// dendro.py:495-499, with the once-raised symbol C1u^l_ab = igt^lm C1_abm).
// cal: CalGt^i = igt^kl C2^i_kl; conn: what stands for it in Ricci, `hat` if
// given (CCZ4).
__device__ __forceinline__ void fold_christoffel(double G[18], const double ig[6], double cal[3], double conn[3],
                                                 const double *hat, double R[6])
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
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int s = 0; s < 6; s++)
            G[6 * k + s] = ig[sym3(k, 0)] * C1[s] + ig[sym3(k, 1)] * C1[6 + s] + ig[sym3(k, 2)] * C1[12 + s];
        cal[k] = sym_dot(ig, &G[6 * k]);
    }
    SGR_STEP;
#pragma unroll
    for (int k = 0; k < 3; k++) conn[k] = hat ? hat[k] : cal[k];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const int i = sym_i(s), j = sym_j(s);
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < 3; k++) v += conn[k] * (C1[6 * i + sym3(j, k)] + C1[6 * j + sym3(i, k)]);
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
// Ricci tensor without its d Gt terms, out T the At equation without them (K:
// its factor of At, K - 2 Theta for CCZ4), lap = igt^ij D_i D_j alpha, aa = At_ij A^ij,
// Gt completed but for d K.
__device__ __forceinline__ void fold_alpha(double T[6], double Gt[3], double &lap, double &AA, const double R[6],
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
        lap = sym_dot(ig, dd);
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
    AA = sym_dot(A, AU);
    const double a3 = 3.0 * alpha * ichi;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double v = 2.0 * alpha * sym_dot(&G[6 * i], AU);
#pragma unroll
        for (int j = 0; j < 3; j++) v -= AU[sym3(i, j)] * (2.0 * da[j] + a3 * dc[j]);
        Gt[i] += v;
    }
}

// First and (want2) pure second derivative along one axis at one point.
__device__ __forceinline__ void axis_derivs(const double *c, int s, int pos, int n, bool lo, bool hi, const AxisConst &a,
                                            bool want2, double &g, double &h)
{
    h = 0.0;
    if (lo || hi) {
        double t[9];
        face_taps(c, s, pos, n, lo, hi, t);
        g = d1_face(t, pos, n, lo, hi, a);
        if (want2) h = d2_face(t, pos, n, lo, hi, a);
    } else {
        double t[7];
#pragma unroll
        for (int o = 0; o < 7; o++) t[o] = c[(o - 3) * s];
        g = d1_int(t + 3, 1, a);
        if (want2) h = d2_int(t + 3, 1, a);
    }
}

// The constraints at one point (GR/constraints.py:161-173) and, PSI4, the real
// and imaginary parts of Psi4 (GR/constraints.py:46-155, with its signs),
// as sums to which each field adds what its derivatives contribute.
template <bool PSI4>
struct Monitor {
    double ham, mom[3], re4, im4;
    double r[3], mr[3], mi[3];  // the tetrad: radial vector, real and imaginary part of m

    // R: Ricci without its d Gt terms; G = C2; dc: d chi; hat: Gt^i
    __device__ __forceinline__ void start(const double R[6], const double G[18], const double g[6], const double ig[6],
                                          double chi, double ichi, double K, const double dc[3], const double A[6],
                                          const double hat[3], double px, double py, double pz)
    {
        double M[9];  // igt^ik A_kj
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++)
                M[3 * i + j] = ig[sym3(i, 0)] * A[sym3(0, j)] + ig[sym3(i, 1)] * A[sym3(1, j)] + ig[sym3(i, 2)] * A[sym3(2, j)];
        double aa = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) aa += M[3 * i + j] * M[3 * j + i];
        ham = chi * sym_dot(ig, R) - aa + (2.0 / 3.0) * K * K;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                v -= hat[k] * A[sym3(i, k)] + 1.5 * ichi * dc[k] * M[3 * k + i];
#pragma unroll
                for (int m = 0; m < 3; m++) v -= G[6 * m + sym3(k, i)] * M[3 * k + m];
            }
            mom[i] = v;
        }
        if constexpr (PSI4) {
            SGR_STEP;
            auto dot = [&](const double a[3], const double b[3]) __attribute__((always_inline)) {
                double v = 0.0;
#pragma unroll
                for (int i = 0; i < 3; i++)
                    v += a[i] * (g[sym3(i, 0)] * b[0] + g[sym3(i, 1)] * b[1] + g[sym3(i, 2)] * b[2]);
                return ichi * v;
            };
            // Gram-Schmidt: r, theta, phi
            double th[3] = {px * pz, py * pz, -(px * px + py * py)}, ph[3] = {-py, px, 0.0};
            r[0] = px, r[1] = py, r[2] = pz;
            const double nr = 1.0 / sqrt(dot(r, r));
#pragma unroll
            for (int i = 0; i < 3; i++) r[i] *= nr;
            const double tt = dot(th, th), rt = dot(r, th), nt = 1.0 / sqrt(tt - rt * rt);
#pragma unroll
            for (int i = 0; i < 3; i++) th[i] = (th[i] - rt * r[i]) * nt;
            const double pp = dot(ph, ph), rp = dot(r, ph), tp = dot(th, ph), np = 1.0 / sqrt(pp - rp * rp - tp * tp);
            const double h2 = 0.70710678118654752440;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                mi[i] = (ph[i] - rp * r[i] - tp * th[i]) * np * h2;
                mr[i] = th[i] * h2;
            }
            SGR_STEP;
            double Ar[3];
#pragma unroll
            for (int i = 0; i < 3; i++) Ar[i] = A[sym3(i, 0)] * r[0] + A[sym3(i, 1)] * r[1] + A[sym3(i, 2)] * r[2];
            auto dot3 = [](const double a[3], const double b[3]) __attribute__((always_inline)) {
                return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
            };
            const double a = ichi * ichi * (dot3(Ar, r) + K * chi * (1.0 / 3.0) + 0.5 * dot3(r, dc));
            double q[6], MM[6], NN[6];
#pragma unroll
            for (int s = 0; s < 6; s++) {
                const int i = sym_i(s), j = sym_j(s);
                q[s] = R[s] + a * A[s];
                MM[s] = mr[i] * mr[j] - mi[i] * mi[j];
                NN[s] = mr[i] * mi[j] + mr[j] * mi[i];
            }
            const double rA = dot3(mr, Ar), iA = dot3(mi, Ar), rd = 0.5 * dot3(mr, dc), jd = 0.5 * dot3(mi, dc);
            re4 = sym_dot(q, MM) - ichi * ichi * (rA * (rA + rd) - iA * (iA + jd));
            im4 = -(sym_dot(q, NN) - ichi * ichi * (rA * (iA - jd) + iA * (rA - rd)));
            SGR_STEP;
            // the connection terms of d_j A_ki + C2^m_ki A_mj
#pragma unroll
            for (int s = 0; s < 6; s++) {
                double W[3];
#pragma unroll
                for (int j = 0; j < 3; j++)
                    W[j] = G[s] * A[sym3(0, j)] + G[6 + s] * A[sym3(1, j)] + G[12 + s] * A[sym3(2, j)];
                curl(s, ichi, W);
            }
        }
    }
    // -1/chi (MR U - NR V) and its imaginary counterpart, from W_kij (j = 0..2)
    // of the symmetric pair s = (k, i)
    __device__ __forceinline__ void curl(int s, double ichi, const double W[3])
    {
        const int k = sym_i(s), i = sym_j(s);
        double vr = 0.0, vi = 0.0;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            double cr = (mr[i] * r[j] - mr[j] * r[i]) * mr[k] - (mi[i] * r[j] - mi[j] * r[i]) * mi[k];
            double ci = (mi[i] * r[j] - mi[j] * r[i]) * mr[k] + (mr[i] * r[j] - mr[j] * r[i]) * mi[k];
            if (k != i) {
                cr += (mr[k] * r[j] - mr[j] * r[k]) * mr[i] - (mi[k] * r[j] - mi[j] * r[k]) * mi[i];
                ci += (mi[k] * r[j] - mi[j] * r[k]) * mr[i] + (mr[k] * r[j] - mr[j] * r[k]) * mi[i];
            }
            vr += cr * W[j];
            vi += ci * W[j];
        }
        re4 -= ichi * vr;
        im4 += ichi * vi;
    }
    __device__ __forceinline__ void add_K(const double d[3])
    {
#pragma unroll
        for (int i = 0; i < 3; i++) mom[i] -= (2.0 / 3.0) * d[i];
    }
    template <int k>
    __device__ __forceinline__ void add_Gt(std::integral_constant<int, k>, const double g[6], double chi, const double d[3])
    {
        ham += chi * d[k];
        if constexpr (PSI4) {
            // R_ij += (g_ki d_j Gt^k + g_kj d_i Gt^k) / 2
            const double gr = g[sym3(k, 0)] * mr[0] + g[sym3(k, 1)] * mr[1] + g[sym3(k, 2)] * mr[2];
            const double gi = g[sym3(k, 0)] * mi[0] + g[sym3(k, 1)] * mi[1] + g[sym3(k, 2)] * mi[2];
            const double dr = mr[0] * d[0] + mr[1] * d[1] + mr[2] * d[2], di = mi[0] * d[0] + mi[1] * d[1] + mi[2] * d[2];
            re4 += gr * dr - gi * di;
            im4 -= gr * di + gi * dr;
        }
    }
    template <int s>
    __device__ __forceinline__ void add_At(std::integral_constant<int, s>, const double ig[6], double ichi, const double d[3])
    {
        constexpr int i = sym_i(s), j = sym_j(s);
        mom[i] += ig[sym3(j, 0)] * d[0] + ig[sym3(j, 1)] * d[1] + ig[sym3(j, 2)] * d[2];
        if (i != j) mom[j] += ig[sym3(i, 0)] * d[0] + ig[sym3(i, 1)] * d[1] + ig[sym3(i, 2)] * d[2];
        if constexpr (PSI4) curl(s, ichi, d);
    }
};

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
// would be waited for with the next LDS access) and read with v_readlane (not in
// a divergent branch, see FieldTable).
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

// What one pass computes: the right-hand side of a system, TVB dissipation added
// to a finished right-hand side (or RK stage), or the constraints
// (with Psi4): gt, chi -> Ricci without d Gt; K, Gt, At -> added to the sums as
// they appear.
enum class Pass { BSSN, CCZ4, TVB3, TVB5, CONSTRAINTS, PSI4 };

// A pass's fields in the order they are processed (those with second
// derivatives first) and where the table of their pointers holds which.
template <Pass PASS>
struct Fields {
    static constexpr bool MONITOR = PASS == Pass::CONSTRAINTS || PASS == Pass::PSI4, CCZ4 = PASS == Pass::CCZ4;
    static constexpr int N = MONITOR ? 17 : CCZ4 ? 25 : 24;   // fields
    static constexpr int ND2 = MONITOR ? 7 : 11;              // with second derivatives
    static constexpr int GT = MONITOR ? 0 : 3, CHI = GT + 6, ALPHA = 10;
    static constexpr int K = MONITOR ? 7 : 11, THETA = 12;
    static constexpr int GAMMA = K + (CCZ4 ? 2 : 1);          // Gt^i (Gamma-hat^i)
    static constexpr int B = GAMMA + 3, AT = MONITOR ? GAMMA + 3 : GAMMA + 6;
    static constexpr int NPV = MONITOR ? 6 : CCZ4 ? 16 : 10;  // point values fetched ahead
    __host__ __device__ static constexpr int field(int p)
    {
        if (p >= GT && p < CHI) return 12 + p - GT;
        if (p == CHI) return 1;
        if (!MONITOR && p < 3) return 6 + p;
        if (!MONITOR && p == ALPHA) return 0;
        if (p == K) return 2;
        if (CCZ4 && p == THETA) return 24;
        if (p < GAMMA + 3) return 3 + p - GAMMA;
        if (p < AT) return 9 + p - B;
        return 18 + p - AT;
    }
    // point value q: shift, gt, alpha (and At); gt alone
    __host__ __device__ static constexpr int pv(int q) { return MONITOR || q < 9 ? q : q == 9 ? ALPHA : AT + q - 10; }
};

// pow, out of line: inlined, its coefficients are hoisted out of the tile loop
// and their registers spill.
__device__ __attribute__((noinline)) double eta_pow(double x, double y) { return pow(x, y); }

// The arrays of the fields in k_rhs's order, one pointer per lane: fetched with
// v_readlane instead of a scalar load with its wait in every field.  Read a
// table (and DescWords) where all lanes are active, never inside a divergent
// branch: if the table's register is spilled, its reload there fills the active
// lanes only, and the pointer may come from a lane that is not.
struct FieldTable {
    int lo, hi;
    __device__ __forceinline__ void set(const double *p) { lo = (int)(uint32_t)(uint64_t)p, hi = (int)((uint64_t)p >> 32); }
    __device__ __forceinline__ SGR_GLOBAL double *get(int p) const
    {
        return (SGR_GLOBAL double *)((uint64_t)(uint32_t)__builtin_amdgcn_readlane(lo, p) |
                                     (uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, p) << 32);
    }
};

// TVB: the characteristic speeds along x, y, z (span nodes each) and the factor
// of the dissipation.
struct TvbArgs {
    const double *lam;
    uint64_t span;
    double sigma;
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
// General shapes share one array: every admissible shape's D_x and D_y (4320
// cells at most) fit twice.  The branch for one that would not (`two`) is never
// taken, but the compiler's schedule without it is 7% slower (blocks of 9 to 33
// points a side, 2.24 -> 2.40 ms).
// The grid is persistent: a workgroup takes every (gridDim.x / 8)-th tile of
// its XCD's range, and the next tile's first fields and point values are
// fetched during the last fields of the current one.  Tiles that reach a
// flagged face run their own copy of the code, the only one with the closure
// forms; `order` lists each range's other tiles first, so that a CU works in
// one copy at a time (both do not fit its instruction cache).
// order: the list's tile numbers, or null for 0, 1, 2, ...
// RK: an RK stage's update instead of the plain RHS (rk.stage >= 0).  ROUND
// (constraints): derivatives rounded to float where the two passes stage them.
// The kernels (k_rhs, ...) are this function; out holds the equations or the
// constraints.
template <Pass PASS, bool UPWIND, bool GEN, bool RK, bool ROUND>
__device__ __forceinline__ void one_pass(const FieldPtrs &in, const OutPtrs &out, const BlockDesc *__restrict__ blocks,
                                         const uint32_t *__restrict__ tile_block, const uint32_t *__restrict__ order,
                                         const Params &P, const RkArgs &rk, const TileRanges &ranges,
                                         const TvbArgs &tv = TvbArgs{})
{
    typedef Fields<PASS> F;
    constexpr bool MONITOR = F::MONITOR, CCZ4 = F::CCZ4, TVB5 = PASS == Pass::TVB5, TVB = TVB5 || PASS == Pass::TVB3;
    constexpr int NT = 512;
    constexpr int RS8 = 24, PS8 = RS8 * TH;       // 8^3: padded halo rows (conflict-free, see k_stencil)
    constexpr int USZ = GEN ? GEN_U_CAP : PS8 * TH;
    constexpr int DXSZ = T * TH * TH, DYSZ = T * T * TH;
    constexpr int DCAP = 4478;                    // general shapes: one buffer of D_x and D_y, what LDS has left
    constexpr int NPF = GEN ? 4 : 3;              // halo loads per thread, 16 bytes each
    __shared__ __align__(16) double U[2 * USZ];
    __shared__ double DX[TVB ? 1 : GEN ? 2 * DCAP : 2 * DXSZ];  // general shapes: DY behind DX
    __shared__ double DY[TVB || GEN ? 1 : 2 * DYSZ];
    __shared__ double DB[MONITOR || TVB ? 1 : 9 * NT];   // each thread's d_j beta^i, at 3 i + j
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
        const int l = t & 63, f = l < F::N ? F::field(l) : 1;
        tin.set(in.p[f]);
        if (MONITOR) {
            tout.set(out.p[l < 6 ? l : 0]);
        } else if (RK) {
            tout.set(rk.acc.p[f]);
            tnext.set(rk.next.p[f]);
            tu0.set(rk.u0.p[f]);
        } else {
            tout.set(out.p[f]);
        }
    }
    // (read from LDS where they are used: scalar loads of them were waited for
    // in every field, registers for them spilled)
    if (!MONITOR && !TVB && t == 0) SP[0] = P.ko_sigma, SP[1] = P.lambda[2], SP[2] = 1.0 - P.lambda[3];

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

    double pv[F::NPV];  // the point's values (Fields::pv) of the tile `aim` points at
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
        if constexpr (TVB) return;
        int lx, ly, lz;
        bool has;
        point_of(thread(), D, lx, ly, lz, has);
        const int o = (lx + GW) + D.n(0) * ((ly + GW) + D.n(1) * (lz + GW));
#pragma unroll
        for (int q = 0; q < F::NPV; q++) pv[q] = (tin.get(F::pv(q)) + lbase)[o];
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
        const int DXZ = TX * HY, DYZ = TX * TY, dy0 = DXZ * (TZ + 2 * GW);
        const bool two = !GEN || dy0 + DYZ * (TZ + 2 * GW) <= DCAP;  // do two of the buffers fit?
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
        // Stores of the points the tile owns.  MASKED: buffer stores from the tile's
        // corner, the other points' offset out of range, which drops the lane.  Behind
        // a branch the number of stores in flight is unknown to the compiler, and each
        // wait for the next field's loads is one for the last field's stores too: 512 x
        // 32^3 7.49 -> 7.28 ms, CCZ4 3% (general shapes 11%).  The general BSSN kernels
        // spill scalar registers over it (33^3 blocks 1.36 -> 1.55 ms) and keep the
        // branch.  (32 bits of offset: a plan with larger planes has no tile lists,
        // stores_reach.)
        constexpr bool MASKED = !GEN || (CCZ4 && !RK);
        const uint64_t corner = tc.i0 + (uint64_t)n0 * (tc.j0 + (uint64_t)n1 * tc.k0);
        uint32_t soff;
        {
            int lx, ly, lz;
            bool has;
            point_of(thread(), D, lx, ly, lz, has);
            const int pi = tc.i0 + lx, pj = tc.j0 + ly, pk = tc.k0 + lz;
            own = has && pi >= tc.oi && pj >= tc.oj && pk >= tc.ok;
            gp = pi + n0 * (pj + n1 * pk);
            soff = own ? 8u * (uint32_t)(lx + n0 * (ly + n1 * lz)) : 0xFFFFFFF8u;
        }
        auto store = [&](SGR_GLOBAL double *a, double k) __attribute__((always_inline)) {
            if constexpr (!MASKED) {
                if (own) a[gp] = k;
                return;
            }
            typedef unsigned Words __attribute__((ext_vector_type(2)));
            const auto r = __builtin_amdgcn_make_buffer_rsrc((void *)(uint64_t)(a + corner), 0, 0xFFFFFFF0u, 0x00027000);
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Words, k), r, (int)soff, 0, 0);
        };
        double bv[3], g[6], ig[6];
#pragma unroll
        for (int d = 0; d < 3; d++) bv[d] = MONITOR ? 0.0 : pv[d];
#pragma unroll
        for (int q = 0; q < 6; q++) g[q] = pv[F::GT + q];
        const double alpha = MONITOR ? 1.0 : pv[MONITOR ? 0 : 9];
        inverse_metric(g, ig);
        double trA3 = 0.0;  // CCZ4: a third of the trace of At
        if constexpr (CCZ4) trA3 = (1.0 / 3.0) * sym_dot(ig, &pv[10]);
        double G[18], R[6], Gt[3], gdb[3], dc[3], div = 0.0, Kv = 0.0, Kr = 0.0, chi = 1.0, eta = 0.0, es = 0.0;
        double hat[3], Zu[3], th = 0.0, Tr = 0.0;  // CCZ4: Gamma-hat, Z^i, Theta, its equation

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
        double A[6];  // At at the point, from field ALPHA on (constraints: CHI)
        auto begin = [&](auto d2_, auto last_, int p, FieldVals &v) __attribute__((always_inline)) {
            constexpr bool D2 = decltype(d2_)::value;
            const int f = F::field(p);
            const int t = thread();
            int lx, ly, lz;
            bool has;
            point_of(t, D, lx, ly, lz, has);
            const int pi = tc.i0 + lx, pj = tc.j0 + ly, pk = tc.k0 + lz;
            if (!MONITOR) v.out = tout.get(p) + obase;
            if (RK) v.next = tnext.get(p) + obase;
            v.face = FACE && !MONITOR && ((lo0 && pi == GW) || (hi0 && pi == n0 - GW - 1) || (lo1 && pj == GW) ||
                                   (hi1 && pj == n1 - GW - 1) || (lo2 && pk == GW) || (hi2 && pk == n2 - GW - 1));
            const int uc = (lx + GW) + RS * (ly + GW) + PS * (lz + GW);
            const int cx = lx + TX * (ly + GW) + DXZ * (lz + GW), cy = lx + TX * ly + DYZ * (lz + GW);
            const double *c = &U[b * USZ + uc];
            double *dx = &DX[GEN ? (two ? b * DCAP : 0) : b * DXSZ], *dy = GEN ? dx + dy0 : &DY[b * DYSZ];
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
            if (D2 && !MONITOR)  // B^k, At_q; K; CCZ4, at alpha: Theta
                v.ex = (tin.get(p < F::CHI ? F::B + p : CCZ4 && p == F::ALPHA ? F::THETA : F::K) + obase)[gp];
            double &g0 = v.g[0], &g1 = v.g[1], &g2 = v.g[2], q0, q1, q2, k0, k1, k2, *h = v.h;
            if constexpr (MONITOR) {
                axis_derivs(c, 1, pi, n0, clo0, chi0, a0, D2, g0, h[0]);
                axis_derivs(c, RS, pj, n1, clo1, chi1, a1, D2, g1, h[3]);
                axis_derivs(c, PS, pk, n2, clo2, chi2, a2, D2, g2, h[5]);
            } else {
                axis_stencils<UPWIND, true>(c, 1, pi, n0, clo0, chi0, bv[0], a0, D2, g0, q0, k0, h[0]);
                axis_stencils<UPWIND, true>(c, RS, pj, n1, clo1, chi1, bv[1], a1, D2, g1, q1, k1, h[3]);
                axis_stencils<UPWIND, true>(c, PS, pk, n2, clo2, chi2, bv[2], a2, D2, g2, q2, k2, h[5]);
            }
            v.uv = c[0];
            if (D2) {
                if (p == (MONITOR ? F::CHI : F::ALPHA)) {
#pragma unroll
                    for (int q = 0; q < 6; q++) A[q] = (tin.get(F::AT + q) + obase)[gp];
                }
                if ((MONITOR && p == F::CHI) || (CCZ4 && p == F::CHI - 1)) {
#pragma unroll
                    for (int k = 0; k < 3; k++) hat[k] = (tin.get(F::GAMMA + k) + obase)[gp];
                }
                if (MONITOR && p == F::CHI) v.ex = (tin.get(F::K) + obase)[gp];
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
            if (D2 && p == (MONITOR ? F::CHI : F::ALPHA)) renew(A, 6);
            if (D2 && ((MONITOR && p == F::CHI) || (CCZ4 && p == F::CHI - 1))) renew(hat, 3);
            // the loads of the field after it (at the end, of the next tile's first;
            // its second: at its start)
            if constexpr (!decltype(last_)::value) {
                keep_dst();
                fetch(p + 2 < F::N ? p + 2 : 0);
            }

            // the terms linear in the field's own advective and KO stencils
            if constexpr (!MONITOR) {
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
                if (!two) __syncthreads();  // DX and DY are read
            }
            if constexpr (ROUND) {
#pragma unroll
                for (int d = 0; d < 3; d++) v.g[d] = (double)(float)v.g[d];
            }
            b ^= 1;
        };
        auto finish_value = [&](const FieldVals &v, double k) __attribute__((always_inline)) {
            SGR_EXACT
            if (!RK) {
                store(v.out, k);
                return;
            }
            const double wk = rk.w * k;
            if (rk.stage == 3) {
                store(v.next, v.acv + wk);
                return;
            }
            store(v.out, (rk.stage == 0 ? v.u0v : v.acv) + wk);
            store(v.next, v.u0v + rk.cn * k);
        };
        auto finish = [&](const FieldVals &v, double alg, double lin) __attribute__((always_inline)) {
            SGR_EXACT
            finish_value(v, v.face ? v.bc : alg + (lin + SP[0] * v.ko));
        };
        auto times = [](double a, double b) __attribute__((always_inline)) {
            SGR_EXACT
            return a * b;
        };
        double *const db = &DB[MONITOR ? 0 : t];
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
            R[q] = -0.5 * (ROUND ? (double)(float)metric_contract(ig, v.h) : metric_contract(ig, v.h));
            if constexpr (MONITOR) return 0.0;
            else return lie_sym(g, db, div, q) - 2.0 * alpha * (CCZ4 ? v.ex - g[q] * trA3 : v.ex);
        };
        auto gamma = [&](auto k_, const FieldVals &v) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value;
            const double ac = alpha * chi;
#pragma unroll
            for (int s = 0; s < 6; s++) {
                const int i = sym_i(s), j = sym_j(s);
                R[s] += ac * (0.5 * (g[sym3(k, i)] * v.g[j] + g[sym3(k, j)] * v.g[i]) - (1.0 / 3.0) * g[s] * v.g[k]);
            }
            if constexpr (CCZ4) {
                Kr += ac * v.g[k];
                Tr += 0.5 * ac * v.g[k];
            }
            const double alg = Gt[k];
            Gt[k] += SP[2] * v.adv;  // what B^k's equation takes of this one
            return alg;
        };

#define SGR_K(n) std::integral_constant<int, n>{}
        const auto yes = std::true_type{};
        const auto no = std::false_type{};
        uint32_t word = tile_of(mnext);
        if constexpr (!MONITOR) {
#pragma unroll 1
            for (int p = 0; p < 3; p++) {  // the shift
                FieldVals v;
                begin(yes, no, p, v);
                if (p == 0) shift(SGR_K(0), v);
                else if (p == 1) shift(SGR_K(1), v);
                else shift(SGR_K(2), v);
            }
            next = first(word);
            word = block_of(next);
        }
#pragma unroll 1
        for (int p = F::GT; p < F::CHI; p++) {  // gt
            FieldVals v;
            begin(yes, no, p, v);
            double alg;
            switch (p - F::GT) {
            case 0: alg = metric(SGR_K(0), v); break;
            case 1: alg = metric(SGR_K(1), v); break;
            case 2: alg = metric(SGR_K(2), v); break;
            case 3: alg = metric(SGR_K(3), v); break;
            case 4: alg = metric(SGR_K(4), v); break;
            default: alg = metric(SGR_K(5), v); break;
            }
            if constexpr (!MONITOR) finish(v, alg, v.adv);
        }
        if constexpr (MONITOR) {
            next = first(word);
            word = block_of(next);
        } else {
            nnext = first(word);
        }
        {
            double cal[3], conn[3];
            fold_christoffel(G, ig, cal, conn, CCZ4 ? hat : nullptr, R);
            if constexpr (!MONITOR)
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    Gt[i] += (2.0 / 3.0) * cal[i] * div -
                             (cal[0] * db[PARK * 3 * i] + cal[1] * db[PARK * (3 * i + 1)] + cal[2] * db[PARK * (3 * i + 2)]);
                    if constexpr (CCZ4) Zu[i] = 0.5 * (hat[i] - cal[i]);
                }
            if constexpr (CCZ4)
#pragma unroll
                for (int i = 0; i < 3; i++)
                    Gt[i] += 2.0 * P.kappa[2] * ((2.0 / 3.0) * Zu[i] * div -
                             (Zu[0] * db[PARK * 3 * i] + Zu[1] * db[PARK * (3 * i + 1)] + Zu[2] * db[PARK * (3 * i + 2)]));
        }
        if constexpr (MONITOR) {
            FieldVals v;
            begin(yes, no, F::CHI, v);
            nnext = first(word);
            Dnext.load(blocks + nnext, thread() & 63);
            chi = v.uv;
            if constexpr (ROUND)
#pragma unroll
                for (int s = 0; s < 6; s++) v.h[s] = (double)(float)v.h[s];
            const double ichi = 1.0 / chi;
            fold_chi(R, G, g, ig, ichi, v.g, v.h);
            Monitor<PASS == Pass::PSI4> M;
            {
                int lx, ly, lz;
                bool has;
                point_of(thread(), D, lx, ly, lz, has);
                const double px = B->pmin[0] + (tc.i0 + lx) * B->ax[0].h, py = B->pmin[1] + (tc.j0 + ly) * B->ax[1].h;
                const double pz = B->pmin[2] + (tc.k0 + lz) * B->ax[2].h;
                M.start(R, G, g, ig, chi, ichi, v.ex, v.g, A, hat, px, py, pz);
            }
#pragma unroll 1
            for (int p = F::K; p < F::N - 2; p++) {  // K, Gt, At
                FieldVals w;
                begin(no, no, p, w);
                switch (p) {
                case F::K: M.add_K(w.g); break;
                case F::GAMMA: M.add_Gt(SGR_K(0), g, chi, w.g); break;
                case F::GAMMA + 1: M.add_Gt(SGR_K(1), g, chi, w.g); break;
                case F::GAMMA + 2: M.add_Gt(SGR_K(2), g, chi, w.g); break;
                case F::AT: M.add_At(SGR_K(0), ig, ichi, w.g); break;
                case F::AT + 1: M.add_At(SGR_K(1), ig, ichi, w.g); break;
                case F::AT + 2: M.add_At(SGR_K(2), ig, ichi, w.g); break;
                default: M.add_At(SGR_K(3), ig, ichi, w.g); break;
                }
            }
            tnc = Dnext.coord(next);
            aim(Dnext, tnc);
            fetch_point(Dnext);
            {
                FieldVals w;
                begin(no, no, F::N - 2, w);
                M.add_At(SGR_K(4), ig, ichi, w.g);
            }
            {
                FieldVals w;
                begin(no, yes, F::N - 1, w);
                M.add_At(SGR_K(5), ig, ichi, w.g);
            }
            // (v_readlane outside the branch: inside it a spilled table would be
            // reloaded for the active lanes only)
            constexpr int NO = PASS == Pass::PSI4 ? 6 : 4;
            SGR_GLOBAL double *o[NO];
#pragma unroll
            for (int q = 0; q < NO; q++) o[q] = tout.get(q) + obase;
            if (own) {
                o[0][gp] = M.ham;
#pragma unroll
                for (int i = 0; i < 3; i++) o[1 + i][gp] = M.mom[i];
                if constexpr (PASS == Pass::PSI4) {
                    o[4][gp] = M.re4;
                    o[5][gp] = M.im4;
                }
            }
        } else {
            {
                FieldVals v;
#pragma unroll 1
                for (int p = F::CHI; p <= F::ALPHA; p++) {
                    begin(yes, no, p, v);
                    if (p == F::CHI) {
                        chi = v.uv;
                        Kv = v.ex;
#pragma unroll
                        for (int d = 0; d < 3; d++) dc[d] = v.g[d];
                        fold_chi(R, G, g, ig, 1.0 / chi, dc, v.h);
                        if constexpr (CCZ4) {  // 2 D_(i Z_j): the chi terms of the physical derivative
                            const double ichi = 1.0 / chi, zd = Zu[0] * dc[0] + Zu[1] * dc[1] + Zu[2] * dc[2];
                            double Zl[3];
#pragma unroll
                            for (int i = 0; i < 3; i++)
                                Zl[i] = g[sym3(i, 0)] * Zu[0] + g[sym3(i, 1)] * Zu[1] + g[sym3(i, 2)] * Zu[2];
#pragma unroll
                            for (int s = 0; s < 6; s++)
                                R[s] += ichi * (Zl[sym_i(s)] * dc[sym_j(s)] + Zl[sym_j(s)] * dc[sym_i(s)] - g[s] * zd);
                        }
                        if (P.eta_func) {
                            const double dd[6] = {dc[0] * dc[0], dc[0] * dc[1], dc[0] * dc[2],
                                                  dc[1] * dc[1], dc[1] * dc[2], dc[2] * dc[2]};
                            es = metric_contract(ig, dd);
                        }
                    } else if (CCZ4) {
                        th = v.ex;
                    }
                    finish(v, p == F::CHI ? (2.0 / 3.0) * chi * (alpha * Kv - div) : -2.0 * alpha * (CCZ4 ? Kv - 2.0 * th : Kv),
                           p == F::CHI ? v.adv : times(P.lambda[0], v.adv));
                }
                if constexpr (CCZ4) {
                    const double k1 = P.kappa[0], k2 = P.kappa[1];
                    const double RZ = chi * sym_dot(ig, R);
                    Tr = 0.5 * alpha * (RZ + (2.0 / 3.0) * Kv * Kv - 2.0 * th * Kv) -
                         chi * (Zu[0] * v.g[0] + Zu[1] * v.g[1] + Zu[2] * v.g[2]) - alpha * k1 * (2.0 + k2) * th;
                    Kr = alpha * (RZ + Kv * Kv - 2.0 * th * Kv) - 3.0 * alpha * k1 * (1.0 + k2) * th;
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        Gt[i] -= 2.0 * th * (ig[sym3(i, 0)] * v.g[0] + ig[sym3(i, 1)] * v.g[1] + ig[sym3(i, 2)] * v.g[2]) +
                                 Zu[i] * alpha * (2.0 * k1 + (4.0 / 3.0) * Kv);
                }
                double Tq[6], lap, aa;
                fold_alpha(Tq, Gt, lap, aa, R, G, g, ig, db, div, alpha, chi, 1.0 / chi, CCZ4 ? Kv - 2.0 * th : Kv, dc, v.g,
                           v.h, A);
                if constexpr (CCZ4) {
                    Kr -= chi * lap;
                    Tr -= 0.5 * alpha * aa;
                } else {
                    Kr = -chi * lap + alpha * ((1.0 / 3.0) * Kv * Kv + aa);
                }
#pragma unroll
                for (int q = 0; q < 6; q++) R[q] = Tq[q];  // from here on the At accumulators
            }
            Dnext.load(blocks + nnext, thread() & 63);
            // CCZ4: K's and Theta's equations take the divergence of Gamma-hat: what
            // they add to it is kept until then
            double kt = 0.0, tt = 0.0;
#pragma unroll 1
            for (int p = F::K; p < F::B; p++) {  // K, (Theta,) Gt
                FieldVals v;
                begin(no, no, p, v);
                double alg;
                switch (p - F::K) {
                case 0:
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        Gt[i] -= (4.0 / 3.0) * alpha *
                                 (ig[sym3(i, 0)] * v.g[0] + ig[sym3(i, 1)] * v.g[1] + ig[sym3(i, 2)] * v.g[2]);
                    alg = Kr;
                    break;
                case F::GAMMA - F::K: alg = gamma(SGR_K(0), v); break;
                case F::GAMMA - F::K + 1: alg = gamma(SGR_K(1), v); break;
                case F::GAMMA - F::K + 2: alg = gamma(SGR_K(2), v); break;
                default:  // Theta
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        Gt[i] += 2.0 * alpha *
                                 (ig[sym3(i, 0)] * v.g[0] + ig[sym3(i, 1)] * v.g[1] + ig[sym3(i, 2)] * v.g[2]);
                    alg = 0.0;
                    break;
                }
                if (CCZ4 && p < F::GAMMA) {
                    SGR_EXACT
                    const double w = v.face ? v.bc : v.adv + SP[0] * v.ko;
                    if (p == F::K) kt = w;
                    else tt = w;
                } else {
                    finish(v, alg, v.adv);
                }
            }
            if constexpr (CCZ4) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int p = F::K + q;
                    FieldVals v;
                    v.ko = 0.0, v.u0v = v.acv = 0.0;
                    v.out = tout.get(p) + obase;
                    if (RK) {
                        v.next = tnext.get(p) + obase;
                        if (rk.stage < 3) v.u0v = (tu0.get(p) + obase)[gp];
                        if (rk.stage > 0) v.acv = v.out[gp];
                    }
                    int lx, ly, lz;
                    bool has;
                    point_of(thread(), D, lx, ly, lz, has);
                    const int pi = tc.i0 + lx, pj = tc.j0 + ly, pk = tc.k0 + lz;
                    v.face = FACE && ((lo0 && pi == GW) || (hi0 && pi == n0 - GW - 1) || (lo1 && pj == GW) ||
                                      (hi1 && pj == n1 - GW - 1) || (lo2 && pk == GW) || (hi2 && pk == n2 - GW - 1));
                    v.bc = q == 0 ? kt : tt;
                    finish_value(v, v.face ? v.bc : (q == 0 ? Kr : Tr) + v.bc);
                }
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
            for (int p = F::B; p < F::N - 2; p++) {  // B, At
                FieldVals v;
                begin(no, no, p, v);
                double alg;
                switch (p - F::B) {
                case 0: alg = Gt[0] - eta * v.uv; break;
                case 1: alg = Gt[1] - eta * v.uv; break;
                case 2: alg = Gt[2] - eta * v.uv; break;
                case 3: alg = R[0]; break;
                case 4: alg = R[1]; break;
                case 5: alg = R[2]; break;
                default: alg = R[3]; break;
                }
                finish(v, alg, p < F::AT ? times(SP[1], v.adv) : v.adv);
            }
            // the last but one fetches for the next tile (the last tile: its own again, unused)
            tnc = Dnext.coord(next);
            aim(Dnext, tnc);
            fetch_point(Dnext);
            {
                FieldVals v;
                begin(no, no, F::N - 2, v);
                finish(v, R[4], v.adv);
            }
            {
                FieldVals v;
                begin(no, yes, F::N - 1, v);
                finish(v, R[5], v.adv);
            }
        }
#undef SGR_K
    };

    // One tile of TVB dissipation (tvb in stencils.h states the forms), added to
    // the outputs.  An axis is pre (W0 X0 - W1 X1 + W2 X2 - ...): the weights W,
    // speeds times coefficients, are the same for every field; X are differences
    // of neighbours (TVB5) or values (TVB3, one-sided forms).  EDGE: a tile with
    // points of the one-sided forms or at a flagged face.
    auto tvb_tile = [&](auto edge_, const DescWords &D, const TileCoord &tc, const ConstBlock B, uint32_t mnext,
                        uint32_t &next, uint32_t &nnext, DescWords &Dnext, TileCoord &tnc) __attribute__((always_inline)) {
        SGR_EXACT
        constexpr bool EDGE = decltype(edge_)::value;
        constexpr int NW = TVB5 ? 6 : 5;
        const int TX = GEN ? D.tdim(0) : T, TY = GEN ? D.tdim(1) : T, TZ = GEN ? D.tdim(2) : T;
        const int HX = TX + 2 * GW, HY = TY + 2 * GW, td[3] = {TX, TY, TZ};
        const int ls[3] = {1, GEN ? HX : RS8, GEN ? HX * HY : PS8};  // strides in U
        const int nn[3] = {D.n(0), D.n(1), D.n(2)}, st[3] = {1, nn[0], nn[0] * nn[1]};
        const uint32_t bflag = D.bflag();
        const uint64_t obase = D.offset();
        int lp[3];
        bool own;
        point_of(thread(), D, lp[0], lp[1], lp[2], own);
        const int pos[3] = {tc.i0 + lp[0], tc.j0 + lp[1], tc.k0 + lp[2]};
        own = own && pos[0] >= tc.oi && pos[1] >= tc.oj && pos[2] >= tc.ok;
        const int gp = pos[0] + nn[0] * (pos[1] + nn[1] * pos[2]);
        const int uc = (lp[0] + GW) * ls[0] + (lp[1] + GW) * ls[1] + (lp[2] + GW) * ls[2];
        double W[3][NW], pre[3];
        bool clo[3], chi_[3];                 // the tile reaches the closures of a flagged face (uniform)
        bool face[3];                         // point of a Kreiss-Oliger closure
        bool head[3], tail[3];                // point of a one-sided form
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int o = d == 0 ? tc.i0 : d == 1 ? tc.j0 : tc.k0;
            clo[d] = EDGE && (bflag >> (2 * d) & 1u) && o < GW + 3;
            chi_[d] = EDGE && (bflag >> (2 * d + 1) & 1u) && o + td[d] - 1 >= nn[d] - GW - 3;
            face[d] = (clo[d] && pos[d] < GW + 3) || (chi_[d] && pos[d] >= nn[d] - GW - 3);
            head[d] = EDGE && TVB5 && !face[d] && pos[d] == GW;
            tail[d] = EDGE && TVB5 && !face[d] && !head[d] && pos[d] == nn[d] - GW - 1;
            pre[d] = TVB5 ? (d == 2 ? B->ax[2].ko_pre : 2.0 / 75.0 / B->ax[d].h) : -1.0 / 12.0 / B->ax[d].h;
            if (EDGE && TVB5) pre[d] = head[d] || tail[d] ? 1.0 / B->ax[d].smr1 : pre[d];
            const SGR_GLOBAL double *l = (const SGR_GLOBAL double *)(uint64_t)(tv.lam + d * tv.span + obase) + gp;
            const int s = st[d];
            if constexpr (!TVB5) {
                W[d][0] = l[-2 * s], W[d][1] = 4.0 * l[-s], W[d][2] = 6.0 * l[0], W[d][3] = 4.0 * l[s], W[d][4] = l[2 * s];
            } else {
                const double l3 = l[tail[d] ? -4 * s : 3 * s], l2 = l[2 * s], l1 = l[s], l0 = l[0];
                const double m1 = l[-s], m2 = l[-2 * s], m3 = l[-3 * s];
                W[d][0] = larger(l3, l2), W[d][1] = 5.0 * larger(l2, l1), W[d][2] = 10.0 * larger(l1, l0);
                W[d][3] = 10.0 * larger(l0, m1), W[d][4] = 5.0 * larger(m1, m2), W[d][5] = larger(m2, m3);
                if (head[d])
                    W[d][0] = l3, W[d][1] = 6.0 * l2, W[d][2] = 15.0 * l1, W[d][3] = 19.0 * l0, W[d][4] = 12.0 * m1,
                    W[d][5] = 3.0 * m2;
                if (tail[d])
                    W[d][0] = l3, W[d][1] = 6.0 * m3, W[d][2] = 15.0 * m2, W[d][3] = 19.0 * m1, W[d][4] = 12.0 * l0,
                    W[d][5] = 3.0 * l1;
            }
        }
        // what is added to: loaded a field ahead, like the halo tile (waited for in
        // its own field, a load waits for the store of the field before as well)
        double av = 0.0, nv = 0.0;
        auto ahead = [&](int p) __attribute__((always_inline)) {
            if (!RK || rk.stage < 3) av = (tout.get(p) + obase)[gp];
            if (RK) nv = (tnext.get(p) + obase)[gp];
        };
        ahead(0);
        auto field = [&](auto last_, int p) __attribute__((always_inline)) {
            SGR_EXACT
            SGR_GLOBAL double *o = tout.get(p) + obase, *nx = RK ? tnext.get(p) + obase : o;
            const double *c = &U[b * USZ + uc];
            const double c0 = c[0];
            uint64_t bp = (uint64_t)B;  // (as in run_tile)
            asm volatile("" : "+s"(bp));
            double Dd[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int s = ls[d];
                if constexpr (!TVB5) {
                    Dd[d] = pre[d] * (W[d][0] * c[-2 * s] - W[d][1] * c[-s] + W[d][2] * c0 - W[d][3] * c[s] + W[d][4] * c[2 * s]);
                } else {
                    double v[7], X[6];
                    // (the one-sided form at the end reads four back: inside the halo,
                    // no tile extent is 1 and the last point is the tile's last)
                    v[0] = c[tail[d] ? -4 * s : 3 * s];
                    v[1] = c[2 * s], v[2] = c[s], v[3] = c0, v[4] = c[-s], v[5] = c[-2 * s], v[6] = c[-3 * s];
#pragma unroll
                    for (int k = 0; k < 6; k++) {
                        X[k] = v[k] - v[k + 1];
                        if constexpr (EDGE) {
                            X[k] = head[d] ? v[k] : X[k];
                            X[k] = tail[d] ? v[k == 0 ? 0 : 7 - k] : X[k];
                        }
                    }
                    Dd[d] = pre[d] * (W[d][0] * X[0] - W[d][1] * X[1] + W[d][2] * X[2] - W[d][3] * X[3] + W[d][4] * X[4] -
                                      W[d][5] * X[5]);
                }
                if (EDGE && (clo[d] || chi_[d])) {
                    double t9[9];
                    face_taps(c, s, pos[d], nn[d], clo[d], chi_[d], t9);
                    const double k = ko_face(t9, pos[d], nn[d], clo[d], chi_[d], axis_of((ConstBlock)bp, d));
                    Dd[d] = face[d] ? k : Dd[d];
                }
            }
            const double a = tv.sigma * ((Dd[0] + Dd[1]) + Dd[2]);
            put(&U[(1 - b) * USZ]);
            double s0 = av + (RK ? rk.w * a : a), s1 = nv + (RK && rk.stage < 3 ? rk.cn * a : rk.w * a);
            asm volatile("" : "+v"(s0), "+v"(s1));  // (formed before the next loads are issued)
            __syncthreads();
            if (p + 1 < F::N) ahead(p + 1);
            if constexpr (!decltype(last_)::value) {
                keep_dst();
                fetch(p + 2 < F::N ? p + 2 : 0);
            }
            if (own) {
                if (!RK || rk.stage < 3) o[gp] = s0;
                if (RK) nx[gp] = s1;
            }
            b ^= 1;
        };
        const auto yes = std::true_type{};
        const auto no = std::false_type{};
        uint32_t word = tile_of(mnext);
#pragma unroll 1
        for (int p = 0; p < 6; p++) field(no, p);
        next = first(word);
        word = block_of(next);
#pragma unroll 1
        for (int p = 6; p < 12; p++) field(no, p);
        nnext = first(word);
        Dnext.load(blocks + nnext, thread() & 63);
#pragma unroll 1
        for (int p = 12; p < F::N - 2; p++) field(no, p);
        tnc = Dnext.coord(next);
        aim(Dnext, tnc);
        field(no, F::N - 2);
        field(yes, F::N - 1);
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
            if (TVB5) face |= o == GW || o + (GEN ? D.tdim(d) : T) >= D.n(d) - GW;  // one-sided forms
        }
        uint32_t next = 0, nnext = 0;
        DescWords Dnext;
        TileCoord tnc;
        const ConstBlock B = (ConstBlock)(uint64_t)(blocks + first(nb));
        if constexpr (TVB) {
            if (face) tvb_tile(std::true_type{}, D, tc, B, mnext, next, nnext, Dnext, tnc);
            else tvb_tile(std::false_type{}, D, tc, B, mnext, next, nnext, Dnext, tnc);
        } else {
            if (face) run_tile(std::true_type{}, D, tc, B, mnext, next, nnext, Dnext, tnc);
            else run_tile(std::false_type{}, D, tc, B, mnext, next, nnext, Dnext, tnc);
        }
        if (m >= end) break;
        tile = next, nb = nnext, D = Dnext, tc = tnc;
    }
}

template <Pass PASS, bool UPWIND, bool GEN, bool RK>
__global__ __launch_bounds__(512, 2) void k_rhs(FieldPtrs in, OutPtrs out, const BlockDesc *__restrict__ blocks,
                                                const uint32_t *__restrict__ tile_block,
                                                const uint32_t *__restrict__ order, Params P, RkArgs rk,
                                                TileRanges ranges)
{
    one_pass<PASS, UPWIND, GEN, RK, false>(in, out, blocks, tile_block, order, P, rk, ranges);
}

// A launch over one list of tiles: its ranges, and at most one workgroup per
// CU, a multiple of 8 so that every XCD's range is served.
inline uint32_t list_grid(const TileList &l, uint32_t grid_cap, TileRanges &r)
{
    uint32_t most = 1;  // tiles of the longest range
    for (int x = 0; x < 9; x++) r.lo[x] = l.lo[x];
    for (int x = 0; x < 8; x++) most = r.lo[x + 1] - r.lo[x] > most ? r.lo[x + 1] - r.lo[x] : most;
    const uint32_t cap = grid_cap < 16 ? 1 : grid_cap / 16;
    return 8 * (most < cap ? most : cap);
}

template <Pass PASS, bool UPWIND, bool GEN, bool RK>
static hipError_t launch_list(const LaunchArgs &a, const TileList &l, hipEvent_t e0, hipEvent_t e1, hipStream_t s)
{
    TileRanges r;
    const uint32_t grid = list_grid(l, a.grid_cap, r);
    hipExtLaunchKernelGGL((k_rhs<PASS, UPWIND, GEN, RK>), dim3(grid), dim3(512), 0, s, e0, e1, 0, a.in, a.out, a.blocks,
                          a.tile_block, l.order, a.params, a.rk, r);
    return hipGetLastError();
}

template <Pass PASS, bool UPWIND, bool RK>
static hipError_t launch_lists(const LaunchArgs &a, hipStream_t s)
{
    const bool fast = a.list[0].lo[8] > a.list[0].lo[0], gen = a.list[1].lo[8] > a.list[1].lo[0];
    hipError_t e = hipSuccess;
    if (fast) e = launch_list<PASS, UPWIND, false, RK>(a, a.list[0], a.ev[0], gen ? nullptr : a.ev[1], s);
    if (e == hipSuccess && gen) e = launch_list<PASS, UPWIND, true, RK>(a, a.list[1], fast ? nullptr : a.ev[0], a.ev[1], s);
    for (int q = 2; q < 4; q++)
        if (e == hipSuccess && a.ev[q]) e = hipEventRecord(a.ev[q], s);
    return e;
}

template <Pass PASS>
static hipError_t launch_pass(const LaunchArgs &a, hipStream_t s)
{
    if (a.rk.stage >= 0) return a.upwind ? launch_lists<PASS, true, true>(a, s) : launch_lists<PASS, false, true>(a, s);
    return a.upwind ? launch_lists<PASS, true, false>(a, s) : launch_lists<PASS, false, false>(a, s);
}

}  // namespace sgr
