// swe_riemann_clear.hpp -- the GeoClaw solvers on clearly subcritical edges.
//
// On most edges of a mesh both cells are wet, the flow is slow against sqrt(g h)
// and the two depths are alike.  There most of geoclaw<SOLVER>
// (swe_riemann.hpp) only confirms what is known beforehand: the middle state's
// speeds do not move the Einfeldt speeds, no sonic test trips, the
// steady-state jump stays inside its bounds, and the first and last wave go
// left and right.  clear_flux evaluates what is left, operation by operation as
// the reference orders it, so its results are geoclaw's bit for bit (up to the
// sign of a zero, which the cell update's sums from +0 absorb).
//
// Clear: with c = sqrt(g h) and U = max(|uL|, |uR|),
//   (cL + cR) / 2 - 2.5 |cL - cR| - U = 3 min(c) - 2 max(c) - U > 0.06,
// and so min(c) - U > 0.06 (rounding moves these by under 1e-7: c < 2^25
// where the test can pass).  Then:
//   - riemanntype: in each of its three structures s1m < 0 < s2m.  Two
//     rarefactions: s1m = uL + 2 cL - 3 sqm with sqm = (2 (cL + cR) - delu) / 4,
//     so s1m <= U + max/2 - 3 min/2 < 0.  Two shocks: the Newton step leaves
//     hm >= h_max, so s1m <= uL - max < 0.  One of each: the secant step leaves
//     hm in [h_min, h_max], so s1m <= U + 2 max - 3 min < 0.  s2m > 0 mirrors
//     this.  sE1 <= uL - cL < 0 < uR + cR <= sE2, so min(sE1, s2m) = sE1 and
//     max(sE2, s1m) = sE2, and neither speed is needed.
//   - the sonic tests: g hbar - U^2 >= min^2 - U^2 > 0.0036, so s1s2bar and
//     s1s2tilde lie below -0.0036, |sE1|, |sE2| > 0.06, and every product
//     compared with criticaltol = 1e-6 is above 1e-5; both pairs of
//     characteristic speeds keep their signs.
//   - the bounds on deldelh are hstar (sE2 - sE1) / sE with
//     hstar = max(N / (sE2 - sE1), 0): they cannot be taken where
//     max(deldelh sE1, deldelh sE2) < (1 - 2^-40) N.  An edge that fails this
//     evaluates them (clear_bounds).
//   - the wave split: sw0 < 0 < sw2, and |sw1| is below the larger of the two.
// The f-wave solver has only the last: min(c) - U > 0.06 is enough for it.
//
// What bounds it: the step kernel is bound by vector issue, and these edges
// are most of a mesh.  A clear edge takes 260 vector instructions (6 of them
// quarter-rate reciprocals and roots), the general solver about 590 with 16
// divisions at 11 instructions each and riemanntype's structures diverging
// within a wave.  The step of the d21 tsunami (4.2 M cells) went from 1404 to
// 806 vector instructions per 64 cells and from 195 to 142 us, that of a d20
// radial dam break from 119 to 65 us.
//
// Divisions: a / b = fma(fma(-b, q, a), r, q), q = a r, with r the reciprocal
// of b to within an ulp (the hardware estimate and two Newton steps): the
// correctly rounded quotient (Markstein) as long as nothing overflows and a is
// 0 or at least 2^-969 (below, the remainder fma(-b, q, a) would round).
// Divisions by one value share one reciprocal, and a cell's is computed once for
// its three edges.  clear_cell keeps out what could overflow or get that small:
// a cell whose momenta or bathymetry are neither 0 nor in [2^-N, 2^60], or
// whose depth is above 2^40, gets a NaN for c, which fails the test on its
// edges.  N = 740 for the augmented solver.  A sum of doubles is 0 or at least
// the last place of its smallest term, and c > 0.06 means g h > 2^-9, so:
//   - u's numerators (the rotated momenta) are 0 or above 2^-795, u above
//     2^-835, uhat's numerator above 2^-893;
//   - if the beds differ, delb > 2^-793 and deldelh's and deldelphi's numerators
//     are above 2^-812.  delphi - deldelphi is 0 or above 2^-855, d0 above
//     2^-847, and the numerators of beta0, beta1 and beta2 are 0 or above 2^-914;
//   - if they do not, deldelh = deldelphi = 0, d0 = hR - hL, and where that is
//     not 0 (then above 2^-73) it exceeds all that is tiny in a numerator.  At
//     equal depths delphi = fl(delhu usum), and beta1's numerator may be anything
//     small; but then f10 = beta0 r20 and f12, of size |delhu| > 2^-849 times
//     l0^2 / span > 2^-34, exceed beta1 < 2^-966 by 2^80 and absorb it.
// The f-wave solver's beta1 is not absorbed where beds are equal and depths differ
// by less than the surface shows: there the numerator is uL uR (hR - hL), and
// N = 340 keeps it above 2^-945.
// (The momenta of a tsunami fall off as its source's Gaussian: with N = 240 for
// both, up to all of the far ocean missed the short path, depending on the
// source's width: over eight sources the d21 step took 144-200 us, now 145-150,
// the d20 adjoint 113-213 us, now 112-117.)
#pragma once

#include "swe_riemann.hpp"

namespace swe {

// 1/x to within an ulp for normal x whose reciprocal is normal.
SWE_HD double rcp_near(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(x);
    double e = __builtin_fma(-x, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, e, r);
#else
    return 1.0 / x;
#endif
}

// a / b correctly rounded, r = rcp_near(b); a, b and the quotient are 0 or
// far from the ends of the exponent range.
SWE_HD double div_near(double a, double b, double r) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
#else
    (void)r;
    return a / b;
#endif
}

// What an edge needs of a cell beside its state: r = 1/h and c = sqrt(g h)
// of a wet cell, 0 for a dry one; c = NaN where the shortcuts must not be taken.
struct ClearCell {
    double r, c;
};

// Gravitational constants the shortcuts are derived for (the whole launch
// takes the general path otherwise).
constexpr double CLEAR_MIN_G = 0x1p-10, CLEAR_MAX_G = 0x1p10;

template <int SOLVER>
SWE_HD ClearCell clear_cell(double eta, double hu, double hv, double b, double drytol, double g) {
    const double h = eta - b;
    ClearCell k{0.0, 0.0};
    if (h > drytol) {
        k.r = rcp_near(h);
        k.c = sqrt_wet(g * h);
    }
    // the exponent of 0 is 0 here, and those of infinities and NaN do not
    // matter: the sum below is not below 2^60 then
    int e;
#if defined(__HIP_DEVICE_COMPILE__)
    e = __builtin_amdgcn_frexp_exp(hu);
    const int e1 = __builtin_amdgcn_frexp_exp(hv), e2 = __builtin_amdgcn_frexp_exp(b);
    // CLEAR_MIN_G <= g < CLEAR_MAX_G by the high words: scalar instructions
    const bool g_fits = (uint32_t)__double2hiint(g) - (uint32_t)__double2hiint(CLEAR_MIN_G) <
                        (uint32_t)__double2hiint(CLEAR_MAX_G) - (uint32_t)__double2hiint(CLEAR_MIN_G);
#else
    int e1, e2;
    (void)frexp(hu, &e);
    (void)frexp(hv, &e1);
    (void)frexp(b, &e2);
    const bool g_fits = g >= CLEAR_MIN_G && g < CLEAR_MAX_G;
#endif
    e = e < e1 ? e : e1;
    e = e < e2 ? e : e2;
    const bool tame = e > (SOLVER == 1 ? -340 : -740) && fabs(hu) + fabs(hv) + fabs(b) < 0x1p60 &&
                      h < 0x1p40 && g_fits;
    if (!tame) k.c = __builtin_nan("");
    return k;
}

// Both sides' normal and tangential momenta and velocities in the edge frame.
struct ClearEdge {
    double pL, qL, pR, qR;  // momenta: normal, tangential
    double uL, vL, uR, vR;
};

SWE_HD ClearEdge clear_edge(double nx, double ny, double hL, double huL, double hvL, double rL,
                            double hR, double huR, double hvR, double rR) {
    ClearEdge e;
    e.pL = nx * huL + ny * hvL;
    e.qL = (-ny) * huL + nx * hvL;
    e.pR = nx * huR + ny * hvR;
    e.qR = (-ny) * huR + nx * hvR;
    e.uL = div_near(e.pL, hL, rL);
    e.uR = div_near(e.pR, hR, rR);
    e.vL = div_near(e.qL, hL, rL);
    e.vR = div_near(e.qR, hR, rR);
    return e;
}

template <int SOLVER>
SWE_HD bool is_clear(double uL, double uR, double cL, double cR) {
    constexpr double K = SOLVER == 1 ? 0.5 : 2.5;
#if defined(__HIP_DEVICE_COMPILE__)
    const double m = __builtin_fma(-K, fabs(cL - cR), 0.5 * (cL + cR));
#else
    const double m = 0.5 * (cL + cR) - K * fabs(cL - cR);
#endif
    return m - fmax(fabs(uL), fabs(uR)) > 0.06;
}

// The bounds on deldelh (riemannsolvers.f:152-164, the subcritical case) of
// an edge near them.
SWE_HD double clear_bounds(double deldelh, double n, double sE1, double sE2) {
    const double hstarHLL = dmax2(n / (sE2 - sE1), 0.0);
    deldelh = dmin2(deldelh, (hstarHLL * (sE2 - sE1)) / sE2);
    return dmax2(deldelh, (hstarHLL * (sE2 - sE1)) / sE1);
}

// edge_flux<SOLVER> on a clear edge (SOLVER 0 or 1).
template <int SOLVER>
SWE_HD void clear_flux(double nx, double ny, const ClearEdge &e, double hL, double bL, double cL,
                       double hR, double bR, double cR, double g, Flux &fL, Flux &fR) {
    static_assert(SOLVER == 0 || SOLVER == 1, "the GeoClaw solvers only");
    const double uL = e.uL, uR = e.uR, vL = e.vL, vR = e.vR;
    const double hsum = hR + hL, usum = uL + uR, delh = hR - hL;
    const double delhu = e.pR - e.pL, delb = bR - bL;
    const double uu = uL * uR;
    const double delphi = ((delhu * usum - uu * delh) + ((0.5 * g) * (((bR + hR) - bL) - hL)) * hsum) -
                          ((0.5 * g) * hsum) * delb;
    const double csum = cR + cL;
    const double uhat = div_near(cL * uL + cR * uR, csum, rcp_near(csum));
    const double chat = sqrt_wet((g * 0.5) * hsum);
    // the operands are finite and not both zero: as dmin2 and dmax2
    const double l0 = fmin(uL - cL, uhat - chat);
    const double l2 = fmax(uR + cR, uhat + chat);
    const double span = l2 - l0, rspan = rcp_near(span);
    double l1 = 0.5 * (l0 + l2);
    double f00, f10, f11, f12, f02;
    if (SOLVER == 1) {  // riemann_fwave, riemannsolvers.f:446-500
        const double deldelphi = -(((g * 0.5) * hsum) * delb);
        const double dec = delphi - deldelphi;
        const double beta1 = div_near(l2 * delhu - dec, span, rspan);
        const double beta2 = div_near(dec - l0 * delhu, span, rspan);
        f00 = beta1;
        f10 = beta1 * l0;
        f11 = 0.0;
        f02 = beta2;
        f12 = beta2 * l2;
    } else {  // riemann_aug_JCP, riemannsolvers.f:2-258
        if (fabs(l1) < 1.0e-20) l1 = 0.0;
        const double hbar = 0.5 * hsum;
        const double ghbar = g * hbar;
        const double s1s2bar = 0.25 * (usum * usum) - ghbar;
        const double s1s2tilde = fmax(0.0, uu) - ghbar;
        const double rbar = rcp_near(s1s2bar);
        const double m = (delb * g) * hbar;
        double deldelh = div_near(m, s1s2bar, rbar);
        const double n = ((e.pL - e.pR) + l2 * hR) - l0 * hL;
        if (!(fmax(deldelh * l0, deldelh * l2) < n * (1.0 - 0x1p-40)))
            deldelh = clear_bounds(deldelh, n, l0, l2);
        double deldelphi = -div_near(m * s1s2tilde, s1s2bar, rbar);
        const double kL = -(hL * delb), kR = -(hR * delb);
        deldelphi = fmin(deldelphi, g * fmax(kL, kR));
        deldelphi = fmax(deldelphi, g * fmin(kL, kR));
        const double d0 = delh - deldelh, d2 = delphi - deldelphi;
        const double r20 = l0 * l0, r22 = l2 * l2;
        // det = -l2 + l0 = -span
        const double beta0 = -div_near(-(d0 * l2) + delhu, span, rspan);
        const double beta1 = -div_near(((delhu * r22 - l2 * d2) - d0 * (l0 * r22 - l2 * r20)) +
                                           (l0 * d2 - delhu * r20),
                                       span, rspan);
        const double beta2 = -div_near(-delhu + d0 * l0, span, rspan);
        f00 = beta0 * l0;
        f10 = beta0 * r20;
        f11 = beta1;
        f02 = beta2 * l2;
        f12 = beta2 * r22;
    }
    const double f20 = f00 * vL, f22 = f02 * vR;
    const double f21 = SOLVER == 1 ? ((e.pR * vR - e.pL * vL) - f20) - f22
                                   : (((hR * uR) * vR - (hL * uL) * vL) - f20) - f22;
    // the middle wave's share of each side: all, none, or half at speed 0
    const double wl = l1 < 0.0 ? 1.0 : (l1 > 0.0 ? 0.0 : 0.5), wr = 1.0 - wl;
    const double nL1 = f10 + wl * f11, nL2 = f20 + wl * f21;
    const double nR1 = wr * f11 + f12, nR2 = wr * f21 + f22;
    const double s = fmax(-l0, l2);
    fL.h = f00;
    fL.hu = nL1 * nx + nL2 * (-ny);
    fL.hv = nL1 * ny + nL2 * nx;
    fL.s = s;
    fR.h = f02;
    fR.hu = nR1 * nx + nR2 * (-ny);
    fR.hv = nR1 * ny + nR2 * nx;
    fR.s = s;
}

}  // namespace swe
