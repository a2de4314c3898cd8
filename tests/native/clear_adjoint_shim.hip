// Host entry point over the reverse of the edge flux on clearly subcritical
// edges and the general one (TEST INFRASTRUCTURE ONLY).
#include "swe_adjoint_clear.hpp"

template <int SOLVER>
static void pairs(long n, const double *nrm, const double *L, const double *R, const double *gfL,
                  const double *gfR, double drytol, double g, double *want, double *got,
                  int8_t *clear) {
    for (long i = 0; i < n; ++i, nrm += 2, L += 4, R += 4, gfL += 3, gfR += 3, want += 8, got += 8) {
        for (int m = 0; m < 8; ++m) want[m] = got[m] = 0.0;
        swe::edge_flux_adj<SOLVER>(nrm[0], nrm[1], L[0], L[1], L[2], L[3], R[0], R[1], R[2], R[3],
                                   drytol, g, 1.0 / (16.0 * g), gfL, gfR, want, want + 4);
        const swe::ClearCell a = swe::clear_cell<SOLVER>(L[0], L[1], L[2], L[3], drytol, g);
        const swe::ClearCell b = swe::clear_cell<SOLVER>(R[0], R[1], R[2], R[3], drytol, g);
        const double hL = L[0] - L[3], hR = R[0] - R[3];
        const swe::ClearEdge e =
            swe::clear_edge(nrm[0], nrm[1], hL, L[1], L[2], a.r, hR, R[1], R[2], b.r);
        clear[i] = swe::is_clear<SOLVER>(e.uL, e.uR, a.c, b.c) &&
                   swe::clear_flux_adj<SOLVER>(nrm[0], nrm[1], e, hL, L[3], a.r, a.c, hR, R[3], b.r,
                                               b.c, g, gfL, gfR, got, got + 4);
    }
}

extern "C" void shim_clear_adjoint(int solver, long n, const double *nrm, const double *L,
                                   const double *R, const double *gfL, const double *gfR,
                                   double drytol, double g, double *want, double *got,
                                   int8_t *clear) {
    (solver == 1 ? pairs<1> : pairs<0>)(n, nrm, L, R, gfL, gfR, drytol, g, want, got, clear);
}
