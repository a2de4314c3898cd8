// Host entry point over the shortcut solver of clearly subcritical edges, so
// that tests can compare it with the general one on the CPU (TEST
// INFRASTRUCTURE ONLY).
#include "swe_riemann_clear.hpp"

template <int SOLVER>
static int both(const double *n, const double *L, const double *R, double drytol, double g,
                double *want, double *got) {
    swe::Flux a, b;
    swe::edge_flux<SOLVER>(n[0], n[1], L[0], L[1], L[2], L[3], R[0], R[1], R[2], R[3], drytol, g,
                           1.0 / (16.0 * g), a, b);
    const double w[8] = {a.h, a.hu, a.hv, a.s, b.h, b.hu, b.hv, b.s};
    for (int i = 0; i < 8; ++i) want[i] = w[i];
    const swe::ClearCell l = swe::clear_cell<SOLVER>(L[0], L[1], L[2], L[3], drytol, g);
    const swe::ClearCell r = swe::clear_cell<SOLVER>(R[0], R[1], R[2], R[3], drytol, g);
    const double hL = L[0] - L[3], hR = R[0] - R[3];
    const swe::ClearEdge e =
        swe::clear_edge(n[0], n[1], hL, L[1], L[2], l.r, hR, R[1], R[2], r.r);
    if (!swe::is_clear<SOLVER>(e.uL, e.uR, l.c, r.c)) return 0;
    swe::clear_flux<SOLVER>(n[0], n[1], e, hL, L[3], l.c, hR, R[3], r.c, g, a, b);
    const double v[8] = {a.h, a.hu, a.hv, a.s, b.h, b.hu, b.hv, b.s};
    for (int i = 0; i < 8; ++i) got[i] = v[i];
    return 1;
}

extern "C" void shim_clear(long count, int solver, const double *n, const double *L,
                           const double *R, double drytol, double g, double *want, double *got,
                           signed char *clear) {
    for (long i = 0; i < count; ++i)
        clear[i] = (signed char)(solver == 1 ? both<1>(n + 2 * i, L + 4 * i, R + 4 * i, drytol, g,
                                                       want + 8 * i, got + 8 * i)
                                             : both<0>(n + 2 * i, L + 4 * i, R + 4 * i, drytol, g,
                                                       want + 8 * i, got + 8 * i));
}
