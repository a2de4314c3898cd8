// swe_adjoint_clear.hpp -- reverse of the edge flux on clearly subcritical
// edges.
//
// Where is_clear (swe_riemann_clear.hpp) holds, edge_flux_adj's branches are
// known: both sides are wet, no wall, the Einfeldt speeds stand (riemanntype's
// reverse gets no seed), nothing is sonic and the first and last wave go left
// and right.  If the steady-state jump also stays clear of its bounds, the
// sweep below is edge_flux_adj's, statement by statement, without the terms
// that are zero: equal to it bit for bit (the sign of a zero aside).  The order
// of its sums is kept because the bathymetry's gradient is a small
// difference of large terms: of the d20 tsunami's, rounding alone is 1e-9.
//
// 368 vector instructions against edge_flux_adj's 1700.
#pragma once

#include "swe_adjoint.hpp"
#include "swe_riemann_clear.hpp"

namespace swe {

// Seeds gfL/gfR on (h, hu, hv) of the left and right fluxes; gradients with
// respect to (eta, hu, hv, b) of both sides.  rL, cL: 1/h and sqrt(g h) of
// clear_cell; e: clear_edge.  Returns false, with nothing valid in the
// gradients, if a bound on the steady-state jump may be taken (WAVE: in any of
// the wave's lanes that are here).
template <int SOLVER, bool WAVE = false>
SWE_HD bool clear_flux_adj(double nx, double ny, const ClearEdge &e, double hL, double bL,
                           double rL, double cL, double hR, double bR, double rR, double cR,
                           double g, const double gfL[3], const double gfR[3], double gQL[4],
                           double gQR[4]) {
    static_assert(SOLVER == 0 || SOLVER == 1, "the GeoClaw solvers only");
    // v only scales f-waves: no correctly rounded division
    const double uL = e.uL, uR = e.uR, vL = e.qL * rL, vR = e.qR * rR;
    const double hsum = hR + hL, usum = uL + uR, uu = uL * uR;
    const double delh = hR - hL, delhu = e.pR - e.pL, delb = bR - bL;
    const double a3 = (0.5 * g) * (((bR + hR) - bL) - hL), c4 = (0.5 * g) * hsum;
    const double delphi = ((delhu * usum - uu * delh) + a3 * hsum) - c4 * delb;
    const double csum = cR + cL, rcsum = rcp_near(csum);
    const double uhat = div_near(cL * uL + cR * uR, csum, rcsum);
    const double chat = sqrt_wet((g * 0.5) * hsum);
    const double a1 = uhat - chat, a2 = uhat + chat, sL = uL - cL, sR = uR + cR;
    const bool selE1 = sL < a1, selE2 = sR > a2;
    const double l0 = selE1 ? sL : a1, l2 = selE2 ? sR : a2;
    const double span = l2 - l0, rspan = rcp_near(span);
    double l1 = 0.5 * (l0 + l2);
    if (SOLVER == 0 && fabs(l1) < 1.0e-20) l1 = 0.0;

    // seeds on the net updates; the middle wave's from the side it goes to
    const double gL0 = gfL[0], gL1 = gfL[1] * nx + gfL[2] * ny, gL2 = -gfL[1] * ny + gfL[2] * nx;
    const double gR0 = gfR[0], gR1 = gfR[1] * nx + gfR[2] * ny, gR2 = -gfR[1] * ny + gfR[2] * nx;
    double gA = l1 < 0.0 ? gL2 : gR2, gB = l1 < 0.0 ? gL1 : gR1;
    if (l1 == 0.0) {
        gA = 0.5 * (gL2 + gR2);
        gB = 0.5 * (gL1 + gR1);
    }
    const double gf20 = gL2 - gA, gf22 = gR2 - gA;

    double ghL, ghR, ghu, guL = 0.0, guR = 0.0, gvL, gvR;  // ghu: of huR, and of -huL
    double ghuL = 0.0, ghuR = 0.0, gdelphi, gdelb, gsE1, gsE2;
    if (SOLVER == 1) {  // riemann_fwave, riemannsolvers.f:446-500
        const double K = (g * 0.5) * hsum;
        const double dec = delphi + K * delb;
        const double beta1 = (l2 * delhu - dec) * rspan, beta2 = (dec - l0 * delhu) * rspan;
        ghuR = gA * vR;
        gvR = gA * e.pR;
        ghuL = -(gA * vL);
        gvL = -(gA * e.pL);
        const double gb2 = gR0 + gR1 * l2 + gf22 * vR;
        gsE2 = gR1 * beta2;
        gvR += gf22 * beta2;
        const double gb1 = gL0 + gL1 * l0 + gf20 * vL;
        gsE1 = gL1 * beta1;
        gvL += gf20 * beta1;
        const double gn2 = gb2 * rspan, gn1 = gb1 * rspan;
        const double gdd = -(gb1 * beta1 + gb2 * beta2) * rspan;
        gdelphi = gn2 - gn1;
        gsE1 -= gn2 * delhu;
        gsE2 += gn1 * delhu;
        ghu = gn1 * l2 - gn2 * l0;
        gsE2 += gdd;
        gsE1 -= gdd;
        gdelb = gdelphi * K;
        ghL = ghR = (gdelphi * delb) * (g * 0.5);
    } else {  // riemann_aug_JCP, riemannsolvers.f:2-258
        const double hbar = 0.5 * hsum, ghbar0 = g * hbar;
        const double s1s2bar = 0.25 * (usum * usum) - ghbar0;
        const bool uneg = 0.0 > uu;
        const double s1s2tilde = (uneg ? 0.0 : uu) - ghbar0;
        const double ib = rcp_near(s1s2bar);
        const double M = (delb * g) * hbar;
        const double deldelh = div_near(M, s1s2bar, ib);
        const double n = ((e.pL - e.pR) + l2 * hR) - l0 * hL;
        bool bounded = !(fmax(deldelh * l0, deldelh * l2) < n * (1.0 - 0x1p-40));
#if defined(__HIP_DEVICE_COMPILE__)
        if (WAVE) bounded = __ballot(bounded) != 0;
#endif
        if (bounded) return false;
        const double Kp = M * s1s2tilde;
        const double p0 = -div_near(Kp, s1s2bar, ib);
        const double pL = -(hL * delb), pR = -(hR * delb);
        const bool hiL = pL > pR, loL = pL < pR;
        const double hi = g * (hiL ? pL : pR), lo = g * (loL ? pL : pR);
        const bool below = p0 < hi;
        const double t2 = below ? p0 : hi;
        const bool above = t2 > lo;
        const double d0 = delh - deldelh, d2 = delphi - (above ? t2 : lo);
        const double r20 = l0 * l0, r22 = l2 * l2, idet = -rspan;
        const double Bq = l0 * r22 - l2 * r20;
        const double beta0 = (-(d0 * l2) + delhu) * idet;
        const double beta1 =
            (((delhu * r22 - l2 * d2) - d0 * Bq) + (l0 * d2 - delhu * r20)) * idet;
        const double beta2 = (-delhu + d0 * l0) * idet;

        // f21 = ((hR uR vR - hL uL vL) - f20) - f22, f22 = f02 vR, f20 = f00 vL
        const double gqR = gA * vR, gqL = -gA * vL;
        gvR = gA * (hR * uR);
        gvL = -(gA * (hL * uL));
        ghR = gqR * uR;
        guR = gqR * hR;
        ghL = gqL * uL;
        guL = gqL * hL;
        const double gf02 = gR0 + gf22 * vR;
        gvR += gf22 * (beta2 * l2);
        const double gf00 = gL0 + gf20 * vL;
        gvL += gf20 * (beta0 * l0);
        // the wave strengths: n0 = -(d0 l2) + d1, n1 = (A - d0 B) + C, n2 = -d1 + d0 l0
        const double gbeta2 = gR1 * r22 + gf02 * l2, gbeta0 = gL1 * r20 + gf00 * l0;
        const double gn0 = gbeta0 * idet, gn1 = gB * idet, gn2 = gbeta2 * idet;
        const double gdet = -(gbeta0 * beta0 + gB * beta1 + gbeta2 * beta2) * idet;
        const double gBq = -gn1 * d0;
        const double gr22 = (gR1 * beta2 + gn1 * delhu) + gBq * l0;
        const double gr20 = (gL1 * beta0 - gBq * l2) - gn1 * delhu;
        gsE2 = (((gf02 * beta2 - gn1 * d2) - gBq * r20) - gn0 * d0) - gdet;
        gsE1 = (((gf00 * beta0 + gn2 * d0) + gBq * r22) + gn1 * d2) + gdet;
        const double gd0 = (gn2 * l0 - gn1 * Bq) - gn0 * l2;
        ghu = ((gn1 * r22 - gn2) - gn1 * r20) + gn0;
        const double gd2 = gn1 * l0 - gn1 * l2;
        gsE2 += (2.0 * l2) * gr22;
        gsE1 += (2.0 * l0) * gr20;
        gdelphi = gd2;
        // the bounds on deldelphi
        const double gt2 = above ? -gd2 : 0.0, glo = above ? 0.0 : -gd2;
        const double gp0 = below ? gt2 : 0.0, ghi = below ? 0.0 : gt2;
        const double xhi = ghi * g, xlo = glo * g;
        const double gpL = (hiL ? xhi : 0.0) + (loL ? xlo : 0.0);
        const double gpR = (hiL ? 0.0 : xhi) + (loL ? 0.0 : xlo);
        ghL -= gpL * delb;
        ghR -= gpR * delb;
        gdelb = -(gpL * hL) - gpR * hR;
        // p0 = -(M s1s2tilde / s1s2bar), deldelh = M / s1s2bar
        const double gKp = -gp0 * ib, gdd = -gd0;
        const double gbar = (gp0 * Kp) * (ib * ib) - (gdd * deldelh) * ib;
        const double gM = gKp * s1s2tilde + gdd * ib, gtilde = gKp * M;
        gdelb += (gM * g) * hbar;
        if (!uneg) {
            guL += gtilde * uR;
            guR += gtilde * uL;
        }
        const double gus = (gbar * 0.5) * usum;
        guL += gus;
        guR += gus;
        const double gh = 0.5 * ((gM * (delb * g) - g * gtilde) - g * gbar);
        ghL = (ghL + gh) - gd0;
        ghR = (ghR + gh) + gd0;
    }
    // the Einfeldt speeds
    const double gsR = selE2 ? gsE2 : 0.0, ga2 = selE2 ? 0.0 : gsE2;
    const double gsL = selE1 ? gsE1 : 0.0, ga1 = selE1 ? 0.0 : gsE1;
    const double guhat = ga1 + ga2, gchat = ga2 - ga1;
    const double gcx = gchat * (0.5 * rcp_near(chat)), gch = gcx * (g * 0.5);
    ghR += gch;
    ghL += gch;
    const double gnum = guhat * rcsum, gden = (-guhat * uhat) * rcsum;
    const double gcL = (gnum * uL + gden) - gsL, gcR = (gnum * uR + gden) + gsR;
    guL = (guL + gnum * cL) + gsL;
    guR = (guR + gnum * cR) + gsR;
    // delphi
    const double gT1 = gdelphi * usum, gu = gdelphi * delhu, gw = -gdelphi * delh;
    guL = (guL + gu) + gw * uR;
    guR = (guR + gu) + gw * uL;
    const double gd = -gdelphi * uu, gE = (gdelphi * hsum) * (0.5 * g), ga = gdelphi * a3;
    const double gc = (-gdelphi * delb) * (0.5 * g);
    ghR = ((ghR + gd) + (ga + gE)) + gc;
    ghL = ((ghL - gd) + (ga - gE)) + gc;
    const double gb = (gdelb + gE) + -gdelphi * c4;  // of bR, and of -bL
    ghuR = (ghuR + ghu) + gT1;
    ghuL = (ghuL - ghu) - gT1;
    ghR += (gcR * g) * (0.5 * rcp_near(cR));
    ghL += (gcL * g) * (0.5 * rcp_near(cL));
    // u = p / h, v = q / h
    ghR = (ghR - (guR * uR) * rR) - (gvR * vR) * rR;
    ghL = (ghL - (guL * uL) * rL) - (gvL * vL) * rL;
    const double gpR = ghuR + guR * rR, gqR = gvR * rR;
    const double gpL = ghuL + guL * rL, gqL = gvL * rL;
    // h = eta - b; p = nx hu + ny hv, q = -ny hu + nx hv
    gQL[0] = ghL;
    gQL[1] = gpL * nx - gqL * ny;
    gQL[2] = gpL * ny + gqL * nx;
    gQL[3] = -gb - ghL;
    gQR[0] = ghR;
    gQR[1] = gpR * nx - gqR * ny;
    gQR[2] = gpR * ny + gqR * nx;
    gQR[3] = gb - ghR;
    return true;
}

}  // namespace swe
