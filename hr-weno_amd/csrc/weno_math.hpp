// weno_math.hpp -- per-cell arithmetic of the WENO -> flux -> divergence -> TVD-stage path.
//
// Two arithmetic forms of the same mathematics are provided, selected by a template flag:
//
//  * Exact  : the reference's own evaluation order, operation for operation (left-to-right
//             sums, (eps+beta)**2 as a product, 12 correctly rounded divides per cell for k=3).
//             The library is compiled with -ffp-contract=off, and a multiply-add is fused only
//             where its product is exact (a power of two), so the results are bit-identical to
//             the reference Fortran built for baseline x86-64.
//  * Fast   : the same formulas with explicit fused multiply-adds and the nonlinear weights
//             consolidated over a common denominator (two divides per cell instead of twelve):
//                 w_r = d_r/q_r / sum_s d_s/q_s  =  d_r*prod_{s!=r} q_s / sum_s d_s*prod_{t!=s} q_t
//             with q_r = (eps+beta_r)**2.  This is an exact rewrite of the algebra; only the
//             rounding differs (a few ulp per reconstruction).  A face's numerator, of the size
//             of beta**4 times a cell value, stays finite for cell-value jumps below ~1e33.
//
// The coefficient tables follow src/hrweno_weno.f90:12-21 (Shu, ICASE 97-65, Table 2.1 and
// eqs. 2.58-2.63).  Window convention: x[K-1+m] holds v_{i+m}, m = -(K-1)..K-1.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define HRW_HD __host__ __device__ __forceinline__
#else
#include <cmath>
#define HRW_HD inline
#endif

namespace hrw {

// --------------------------------------------------------------------------------------
// Tables (src/hrweno_weno.f90:12-21).  C<K>::c[r+1][j] == c(j, r).
template <int K> struct Tab;
template <> struct Tab<1> {
    static constexpr double d[1] = {1.0};
    static constexpr double c[2][1] = {{1.0}, {1.0}};
};
template <> struct Tab<2> {
    static constexpr double d[2] = {2.0 / 3, 1.0 / 3};
    static constexpr double c[3][2] = {{3.0 / 2, -1.0 / 2}, {1.0 / 2, 1.0 / 2}, {-1.0 / 2, 3.0 / 2}};
};
template <> struct Tab<3> {
    static constexpr double d[3] = {0.3, 0.6, 0.1};
    static constexpr double c[4][3] = {{11.0 / 6, -7.0 / 6, 1.0 / 3},
                                       {1.0 / 3, 5.0 / 6, -1.0 / 6},
                                       {-1.0 / 6, 5.0 / 6, 1.0 / 3},
                                       {1.0 / 3, -7.0 / 6, 11.0 / 6}};
};

HRW_HD double fma_(double a, double b, double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_fma(a, b, c);
#else
    return std::fma(a, b, c);
#endif
}

// --------------------------------------------------------------------------------------
// Smoothness indicators, src/hrweno_weno.f90:183-204 (eqs. 2.62, 2.63), reference order.
template <int K> HRW_HD void beta_exact(const double *x, double *beta)
{
    const double *v = x + (K - 1);   // v[m] = v_{i+m}
    if constexpr (K == 1) {
        beta[0] = 0.0;
    } else if constexpr (K == 2) {
        double a = v[1] - v[0];
        double b = v[0] - v[-1];
        beta[0] = a * a;
        beta[1] = b * b;
    } else {
        double a, b;
        a = (v[0] - 2 * v[1]) + v[2];
        b = (3 * v[0] - 4 * v[1]) + v[2];
        beta[0] = 13.0 / 12 * (a * a) + 1.0 / 4 * (b * b);
        a = (v[-1] - 2 * v[0]) + v[1];
        b = v[-1] - v[1];
        beta[1] = 13.0 / 12 * (a * a) + 1.0 / 4 * (b * b);
        a = (v[-2] - 2 * v[-1]) + v[0];
        b = (v[-2] - 4 * v[-1]) + 3 * v[0];
        beta[2] = 13.0 / 12 * (a * a) + 1.0 / 4 * (b * b);
    }
}

// 1/x to within a fraction of an ulp: hardware estimate (2^-24.4) and two Newton steps.
#if defined(__HIPCC__)
__device__ __forceinline__ double rcp_nr(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = fma_(-x, r, 1.0);
    r = fma_(r, e, r);
    e = fma_(-x, r, 1.0);
    return fma_(r, e, r);
}

// n/d correctly rounded, given y = rcp_nr(d): the quotient estimate n*y is within an ulp, its
// remainder n - d*q is exact in one fused operation, and one correction rounds it (Markstein,
// "Computation of elementary functions on the IBM RISC System/6000", 1990).  That is the IEEE
// quotient while no intermediate leaves the normal range: |n| and d between 2^-900 and 2^900,
// their exponents less than 768 apart (n = +0 is exact too; -0 gives +0).
__device__ __forceinline__ double quot(double n, double d, double y)
{
    const double q = n * y;
    return fma_(fma_(-d, q, n), y, q);
}
#endif

// The nonlinear weights of the right (w) and left (wt) faces from the smoothness indicators,
// src/hrweno_weno.f90:206-214: alfa_r = d_r/(eps + beta_r)**2, w_r = alfa_r/sum(alfa).  Every
// quotient is the correctly rounded one; on the device the quotients over one denominator share
// its reciprocal (5 reciprocals and 11 quotients for k = 3, about 60 operations instead of the
// 120 of the divides), which needs sum (eps + beta_r)**2 < 2^400 -- with eps > 2^-52 every
// operand of a quotient then lies in (2^-405, 2^400).  Larger or NaN indicators take the divides.
template <int K> HRW_HD void weights_exact(const double *beta, double eps, double *w, double *wt)
{
    if constexpr (K == 1) {
        w[0] = wt[0] = 1.0;   // alfa/alfa
        return;
    } else {
        double q[K], alfa[K], alfat[K];
        double qs = 0.0;
#pragma unroll
        for (int r = 0; r < K; ++r) {
            q[r] = eps + beta[r];
            q[r] = q[r] * q[r];
            qs += q[r];
        }
#if defined(__HIP_DEVICE_COMPILE__)
        if (qs < 0x1p400) {
#pragma unroll
            for (int r = 0; r < K; ++r) {
                const double y = rcp_nr(q[r]);
                alfa[r] = quot(Tab<K>::d[r], q[r], y);
                alfat[r] = 2 * r == K - 1 ? alfa[r] : quot(Tab<K>::d[K - 1 - r], q[r], y);
            }
            double sa = alfa[0], sat = alfat[0];
#pragma unroll
            for (int r = 1; r < K; ++r) {
                sa = sa + alfa[r];
                sat = sat + alfat[r];
            }
            const double ya = rcp_nr(sa), yt = rcp_nr(sat);
#pragma unroll
            for (int r = 0; r < K; ++r) {
                w[r] = quot(alfa[r], sa, ya);
                wt[r] = quot(alfat[r], sat, yt);
            }
            return;
        }
#endif
#pragma unroll
        for (int r = 0; r < K; ++r) {
            alfa[r] = Tab<K>::d[r] / q[r];
            alfat[r] = Tab<K>::d[K - 1 - r] / q[r];
        }
        double sa = 0.0, sat = 0.0;
#pragma unroll
        for (int r = 0; r < K; ++r) sa = sa + alfa[r];
#pragma unroll
        for (int r = 0; r < K; ++r) sat = sat + alfat[r];
#pragma unroll
        for (int r = 0; r < K; ++r) {
            w[r] = alfa[r] / sa;
            wt[r] = alfat[r] / sat;
        }
    }
}

// Exact form of one cell, src/hrweno_weno.f90:176-214.  ci == nullptr: uniform tables;
// otherwise ci[(r+1)*K + j] == cnu(j, r, i) (non-uniform grid, eq. 2.20).
template <int K> HRW_HD void weno_cell_exact(const double *x, double eps, const double *ci,
                                             double &vl, double &vr)
{
    const double *v = x + (K - 1);
    double vrr[K], vlr[K], beta[K], w[K], wt[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        double s = 0.0, sl = 0.0;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const double cr = ci ? ci[(r + 1) * K + j] : Tab<K>::c[r + 1][j];
            s = s + cr * v[-r + j];
        }
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const double cl = ci ? ci[r * K + j] : Tab<K>::c[r][j];
            sl = sl + cl * v[-r + j];
        }
        vrr[r] = s;
        vlr[r] = sl;
    }
    beta_exact<K>(x, beta);
    weights_exact<K>(beta, eps, w, wt);
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int r = 0; r < K; ++r) a = a + w[r] * vrr[r];
#pragma unroll
    for (int r = 0; r < K; ++r) b = b + wt[r] * vlr[r];
    vr = a;
    vl = b;
}

// Pieces of the triple (a, b, c) = (v_m, v_m+1, v_m+2) that the K = 3 reconstructions of cells
// m, m+1 and m+2 draw on, in either arithmetic form: the smoothness indicators beta_0(m),
// beta_1(m+1), beta_2(m+2) and the four candidates c(:,r).T, r = -1..2 (vlr0(m), vrr0(m) =
// vlr1(m+1), vrr1(m+1) = vlr2(m+2), vrr2(m+2)).  FAST keeps 12 beta and 6 c.T.
struct Tri3 {
    double bA, bB, bC;
    double Pm, P0, P1, P2;
};

// EXACT: each piece is what beta_exact and weno_cell_exact form for those cells, operation for
// operation (a product by 2 or 1/4 is exact, so fusing it with the sum it enters changes nothing;
// where 2b overflows, 4b does too, which leaves no finite indicator either way, but 4b may overflow
// alone, so it is not fused); formed once and used by three cells.
HRW_HD Tri3 tri3_exact(double a, double b, double c)
{
    Tri3 t;
    const double D = fma_(-2.0, b, a) + c;
    const double dd = 13.0 / 12 * (D * D);
    const double b4 = 4 * b;
    const double b0 = (3 * a - b4) + c;
    const double b1 = a - c;
    const double b2 = (a - b4) + 3 * c;
    t.bA = fma_(0.25, b0 * b0, dd);
    t.bB = fma_(0.25, b1 * b1, dd);
    t.bC = fma_(0.25, b2 * b2, dd);
    auto cand = [&](const double *q) { return (fma_(q[0], a, 0.0) + q[1] * b) + q[2] * c; };
    t.Pm = cand(Tab<3>::c[0]);
    t.P0 = cand(Tab<3>::c[1]);
    t.P1 = cand(Tab<3>::c[2]);
    t.P2 = cand(Tab<3>::c[3]);
    return t;
}
// One reconstruction from T(i-2), T(i-1), T(i): weno_cell_exact<3> from the shared pieces.
HRW_HD void recon3_exact(double eps, const Tri3 &t2, const Tri3 &t1, const Tri3 &t0, double &vl,
                         double &vr)
{
    const double beta[3] = {t0.bA, t1.bB, t2.bC};
    double w[3], wt[3];
    weights_exact<3>(beta, eps, w, wt);
    vr = (fma_(w[0], t0.P0, 0.0) + w[1] * t1.P1) + w[2] * t2.P2;
    vl = (fma_(wt[0], t0.Pm, 0.0) + wt[1] * t1.P0) + wt[2] * t2.P1;
}

// The same of a pair (a, b) = (v_m, v_m+1) for K = 2: beta_0(m) = beta_1(m+1), and the
// candidates S = vrr0(m) = vlr1(m+1), Rr = vrr1(m+1), Lr = vlr0(m) (FAST keeps twice those).
struct Pair2 {
    double B, S, Rr, Lr;
};
HRW_HD Pair2 pair2_exact(double a, double b)
{
    Pair2 p;
    const double d = b - a;
    p.B = d * d;
    auto cand = [&](const double *q) { return fma_(q[0], a, 0.0) + q[1] * b; };
    p.Lr = cand(Tab<2>::c[0]);
    p.S = cand(Tab<2>::c[1]);
    p.Rr = cand(Tab<2>::c[2]);
    return p;
}
HRW_HD void recon2_exact(double eps, const Pair2 &p1, const Pair2 &p0, double &vl, double &vr)
{
    const double beta[2] = {p0.B, p1.B};
    double w[2], wt[2];
    weights_exact<2>(beta, eps, w, wt);
    vr = fma_(w[0], p0.S, 0.0) + w[1] * p1.Rr;
    vl = fma_(wt[0], p0.Lr, 0.0) + wt[1] * p1.S;
}

// The faces nr/sr, nl/sl by quot; `out` is set where that is not the correctly rounded quotient (or an
// ulp off it, where the numerator lies below 2^-900): the sums lie above 2^-210 for eps > 2^-52 and
// within a factor 3 of each other, so their reciprocals are normal numbers while sr < 2^1020, and a
// numerator that has overflowed (jumps above some 1e33) gives NaN.  DIVIDE: the divide.
template <bool DIVIDE>
HRW_HD void fast_faces(double nr, double sr, double nl, double sl, double &vl, double &vr, bool &out)
{
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (!DIVIDE) {
        vr = quot(nr, sr, rcp_nr(sr));
        vl = quot(nl, sl, rcp_nr(sl));
        out = out | __builtin_isunordered(vr, vl) | !(sr < 0x1p1020);
        return;
    }
#endif
    (void)out;
    vr = nr / sr;
    vl = nl / sl;
}

// Fast form of one cell on a uniform grid (see the header comment), its faces by fast_faces.
template <int K, bool DIVIDE>
HRW_HD void weno_cell_fast(const double *x, double eps, double &vl, double &vr, bool &out)
{
    const double *v = x + (K - 1);
    if constexpr (K == 1) {
        vr = v[0];
        vl = v[0];
    } else if constexpr (K == 2) {
        // candidates: vrr0=(v0+v1)/2, vrr1=(-v-1+3v0)/2, vlr0=(3v0-v1)/2, vlr1=(v-1+v0)/2
        const double a = v[1] - v[0], b = v[0] - v[-1];
        double q0 = eps + a * a;
        double q1 = eps + b * b;
        q0 = q0 * q0;
        q1 = q1 * q1;
        // w_r ~ d_r / q_r  ->  weights proportional to d_0*q1, d_1*q0
        const double ar0 = (2.0 / 3) * q1, ar1 = (1.0 / 3) * q0;
        const double al0 = (1.0 / 3) * q1, al1 = (2.0 / 3) * q0;
        const double vrr0 = 0.5 * (v[0] + v[1]);
        const double vrr1 = fma_(1.5, v[0], -0.5 * v[-1]);
        const double vlr0 = fma_(1.5, v[0], -0.5 * v[1]);
        const double vlr1 = 0.5 * (v[-1] + v[0]);
        fast_faces<DIVIDE>(fma_(ar0, vrr0, ar1 * vrr1), ar0 + ar1, fma_(al0, vlr0, al1 * vlr1), al0 + al1, vl, vr, out);
    } else {
        const double vm2 = v[-2], vm1 = v[-1], v0 = v[0], vp1 = v[1], vp2 = v[2];
        // candidate stencils, c3 rows r+1 (right faces) and r (left faces)
        const double vrr0 = fma_(-1.0 / 6, vp2, fma_(5.0 / 6, vp1, (1.0 / 3) * v0));
        const double vrr1 = fma_(1.0 / 3, vp1, fma_(5.0 / 6, v0, (-1.0 / 6) * vm1));
        const double vrr2 = fma_(11.0 / 6, v0, fma_(-7.0 / 6, vm1, (1.0 / 3) * vm2));
        const double vlr0 = fma_(1.0 / 3, vp2, fma_(-7.0 / 6, vp1, (11.0 / 6) * v0));
        const double vlr1 = fma_(-1.0 / 6, vp1, fma_(5.0 / 6, v0, (1.0 / 3) * vm1));
        const double vlr2 = fma_(1.0 / 3, v0, fma_(5.0 / 6, vm1, (-1.0 / 6) * vm2));
        // smoothness indicators (eq. 2.63)
        double a, b;
        a = fma_(-2.0, vp1, v0) + vp2;
        b = fma_(-4.0, vp1, fma_(3.0, v0, vp2));
        const double b0 = fma_(13.0 / 12 * a, a, 0.25 * (b * b));
        a = fma_(-2.0, v0, vm1) + vp1;
        b = vm1 - vp1;
        const double b1 = fma_(13.0 / 12 * a, a, 0.25 * (b * b));
        a = fma_(-2.0, vm1, vm2) + v0;
        b = fma_(3.0, v0, fma_(-4.0, vm1, vm2));
        const double b2 = fma_(13.0 / 12 * a, a, 0.25 * (b * b));
        double q0 = eps + b0, q1 = eps + b1, q2 = eps + b2;
        q0 = q0 * q0;
        q1 = q1 * q1;
        q2 = q2 * q2;
        const double m0 = q1 * q2, m1 = q0 * q2, m2 = q0 * q1;
        // right face: d = (0.3, 0.6, 0.1); left face: reversed d = (0.1, 0.6, 0.3)
        const double sr = fma_(0.3, m0, fma_(0.6, m1, 0.1 * m2));
        const double sl = fma_(0.1, m0, fma_(0.6, m1, 0.3 * m2));
        const double nr = fma_(0.3 * m0, vrr0, fma_(0.6 * m1, vrr1, (0.1 * m2) * vrr2));
        const double nl = fma_(0.1 * m0, vlr0, fma_(0.6 * m1, vlr1, (0.3 * m2) * vlr2));
        fast_faces<DIVIDE>(nr, sr, nl, sl, vl, vr, out);
    }
}
template <int K> HRW_HD void weno_cell_fast(const double *x, double eps, double &vl, double &vr)
{
    bool out = false;
    weno_cell_fast<K, false>(x, eps, vl, vr, out);
    if (out) weno_cell_fast<K, true>(x, eps, vl, vr, out);
}

// --------------------------------------------------------------------------------------
// Numerical fluxes, src/hrweno_fluxes.f90:42-43 and :66-74, given fm=f(vm), fp=f(vp).
HRW_HD double lax_friedrichs(double fm, double fp, double vm, double vp, double alpha)
{
    return ((fm + fp) - alpha * (vp - vm)) / 2;
}
HRW_HD double godunov(double fm, double fp, double vm, double vp)
{
    if (vm <= vp) return fm < fp ? fm : fp;
    return fm > fp ? fm : fp;
}

// Burgers f(v) = v**2/2 (example/example1_burgers_1d_fv.f90:120)
HRW_HD double burgers_f(double v) { return (v * v) / 2; }

enum NumFlux : int { LF = 0, GODUNOV = 1 };

template <int FLUX, bool FAST>
HRW_HD double burgers_numflux(double vm, double vp, double alpha)
{
    if constexpr (FLUX == GODUNOV) {
        return godunov(burgers_f(vm), burgers_f(vp), vm, vp);
    } else if constexpr (FAST) {
        // ((vm^2 + vp^2)/2 - alpha*(vp-vm)) / 2
        return fma_(0.25, fma_(vm, vm, vp * vp), (-0.5 * alpha) * (vp - vm));
    } else {
        return lax_friedrichs(burgers_f(vm), burgers_f(vp), vm, vp, alpha);
    }
}

// Linear flux (a + b*x)*v (example/example2_pbe_2d_fv.f90:131-155 with a growth rate g(x)).
// The coefficient is formed without contraction in both forms so that g(x) is the
// reference's value exactly.
HRW_HD double linear_coef(double a, double b, double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __dadd_rn(a, __dmul_rn(b, x));
#else
    return a + b * x;
#endif
}

// Edge i of a linear grid, xmin + rx*i (src/hrweno_grids.f90:76-78), never contracted.
HRW_HD double linear_edge(double xmin, double rx, long long i)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __dadd_rn(xmin, __dmul_rn(rx, (double)i));
#else
    return xmin + rx * (double)i;
#endif
}
// The same for 32-bit indices (one conversion instruction instead of four).
HRW_HD double linear_edge32(double xmin, double rx, int i)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __dadd_rn(xmin, __dmul_rn(rx, (double)i));
#else
    return xmin + rx * (double)i;
#endif
}

// x/3 correctly rounded except in rare ties, from one multiply and two FMAs.
HRW_HD double div3_fast(double x)
{
    const double inv3 = 1.0 / 3;
    double q = x * inv3;
    double r = fma_(-3.0, q, x);
    return fma_(r, inv3, q);
}

// --------------------------------------------------------------------------------------
// TVD stage combinations, src/hrweno_tvdode.f90:139,150-152,163-167 and :257.
// u0 = state at the start of the step, us = stage input, L = rhs(us), h = dt.
enum Stage : int {
    RK1 = 0,     // u  = u + dt*L(u)
    RK2_1 = 1,   // ui = u + dt*L(u)
    RK2_2 = 2,   // u  = (u + ui + dt*L(ui))/2
    RK3_1 = 3,   // ui = u + dt*L(u)
    RK3_2 = 4,   // ui = (3u + ui + dt*L(ui))/4
    RK3_3 = 5,   // u  = (u + 2ui + 2dt*L(ui))/3
    MS3 = 6      // ui = (25u + 50dt*L(u) + 7u_{n-4} + 10dt*L(u_{n-4}))/32
};

template <bool FAST>
HRW_HD double stage_update(int stage, double u0, double us, double L, double h, double uo4,
                           double Lo4)
{
    switch (stage) {
    case RK1:
    case RK2_1:
    case RK3_1:
        return FAST ? fma_(h, L, us) : us + h * L;
    case RK2_2:
        return FAST ? 0.5 * fma_(h, L, u0 + us) : ((u0 + us) + h * L) / 2;
    case RK3_2:
        return FAST ? 0.25 * fma_(h, L, fma_(3.0, u0, us)) : ((3 * u0 + us) + h * L) / 4;
    case RK3_3:
        return FAST ? div3_fast(fma_(2.0 * h, L, fma_(2.0, us, u0)))
                    : ((u0 + 2 * us) + (2 * h) * L) / 3;
    default:  // MS3
        return FAST ? 0.03125 * fma_(10.0 * h, Lo4, fma_(7.0, uo4, fma_(50.0 * h, L, 25.0 * us)))
                    : ((((25 * us) + (50 * h) * L) + 7 * uo4) + (10 * h) * Lo4) / 32;
    }
}

}  // namespace hrw
