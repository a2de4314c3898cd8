// swe_step.hip -- the fused SWE Euler step for gfx950 (MI355X).
//
// One step kernel performs one traversal of SWE_euler_timestep.f90 over
// every mesh of a batch: the GeoClaw flux on every edge (skeleton_scalar_op
// :196-215 and bnd_skeleton_scalar_op :231-255), the cell update with the
// wet/dry limiter (cell_update_op :257-284, volume_op :307-355) and each
// chunk's CFL / refinement partials.  The partials of a scenario are reduced,
// and the dt chain advanced (post_traversal_grid_op :111-131,
// pre_traversal_grid_op :89-109), in one of three ways: by the next step of a
// chain of them (CHAIN_CHUNKS), by the last workgroup to meet the others
// (MEET_CHUNKS), or by a small finalize kernel.
//
// Mapping.  A workgroup processes chunks of CH consecutive SFC cells of one
// scenario.  It stages the chunk's state in LDS with a compact list of the edges
// it must solve (each edge inside the chunk once, from its left side; edges to
// cells outside the chunk and domain-boundary edges by this chunk), which is
// stored with the mesh or built here, solves them with one thread per list entry, scatters
// both sides' fluxes into LDS, then updates its cells and reduces the CFL
// candidate.  The Sierpinski order keeps almost every neighbour inside the
// chunk, so ~1.6 Riemann solves per cell are done instead of 3, and halo
// reads are L2 hits.  The edges that leave the chunk come last in the list: the
// waves of inner edges neither wait for halo reads nor exchange the sides.
// A wave whose edges are all clearly subcritical takes the short solver of
// swe_riemann_clear.hpp (same results); the others are solved in a second
// pass over the list.  Chunks are dealt to XCDs in contiguous SFC ranges so
// each XCD's L2 holds the halos of its own chunks; a grid smaller than the
// chunk count makes the launch persistent (grid-stride).
//
// NT threads work on a chunk, CH or 2 CH; the first CH hold a cell each.
//
// Edge semantics (Tools_adaptive_traversal.f90:606-640).  The left state of
// an interior edge is the cell that touches it first in the current
// traversal direction: the lower SFC index when forward, the higher when
// backward; the edge normal is the left cell's outward normal.  The two cells
// of an edge see bit-identical normals of opposite sign, so each cell uses
// its own table entry and negates it when it is the right cell.  The update
// sums fluxes in the reference edge-index order of the traversal: edges
// 1,2,3 of the forward plotter type, or 3,2,1 when the cells are reversed
// (SFC_data_types.f90:473-486 negates the plotter type, swapping the legs).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "swe_device.hpp"
#include "swe_finalize.hpp"
#include "swe_internal.hpp"
#include "swe_riemann.hpp"
#include "swe_riemann_clear.hpp"
#include "swe_riemann_tol.hpp"

namespace swe {

__constant__ double c_normal[17 * 3 * 2];  // [plotter + 8][edge][x,y]
__constant__ double c_leg[64];             // l(k) = sqrt(0.5)**k at k + 1

// One workgroup's partials meet the others' (cl: its chunk among the n of the
// scenario).  Returns true in the last one, with the scenario's values.
// Relaxed device-wide atomics in program order: each returns before the next
// is issued (the empty asm needs its result).
__device__ __forceinline__ bool meet(Meet *f, uint32_t cl, uint32_t n, double &fastest,
                                     long long &refined) {
    auto bits = (unsigned long long)__double_as_longlong(fastest);
    unsigned long long inc = 1ull | ((unsigned long long)refined << 32);
    auto come = [&](Meet *m, uint32_t expected) -> bool {
        const unsigned long long seen = __hip_atomic_fetch_max(&m->fastest, bits, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::"v"(seen) : "memory");
        const unsigned long long old =
            __hip_atomic_fetch_add(&m->came, inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)old + 1u != expected) return false;
        asm volatile("" ::: "memory");
        bits = __hip_atomic_exchange(&m->fastest, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&m->came, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        inc = 1ull | (((old >> 32) + (inc >> 32)) << 32);
        return true;
    };
    if (n > MEET_FAN) {
        const uint32_t k = cl % MEET_FAN;
        if (!come(f + 1 + k, (n - k + MEET_FAN - 1) / MEET_FAN)) return false;
        if (!come(f, MEET_FAN)) return false;
    } else if (!come(f, n)) {
        return false;
    }
    fastest = __longlong_as_double((long long)bits);
    refined = (long long)(inc >> 32);
    return true;
}

// Four waves per SIMD (at most 128 VGPRs, a few spilled) outrun three
// unspilled ones: the LDS of four 256-cell workgroups fits a CU.
// JUMPS: the refinement flags follow the elevation-jump criterion
// (StepArgs::flag_jumps); a template parameter so that the plain kernel's
// code and registers do not pay for it.  RAW: one mesh (StepArgs::scen0)
// whose nbr holds plain neighbour cells (StepArgs::raw_nbr).  TOL: the
// toleranced arithmetic of swe_riemann_tol.hpp (StepArgs::tol; the GeoClaw
// solvers only): the chunk stages each cell's depth, world velocity,
// bathymetry and sqrt(g h) instead of its state and keeps its own state in
// registers.
template <int SOLVER, int CH, int NT, bool JUMPS, bool RAW = false, bool TOL = false>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void euler_step_kernel(
    StepArgs args) {
    static_assert(!(RAW && TOL), "the toleranced kernel reads packed neighbours");
    constexpr bool GEOCLAW = SOLVER == 0 || SOLVER == 1;
    static_assert(!TOL || GEOCLAW, "toleranced GeoClaw solvers only");
    constexpr bool CLEAR = GEOCLAW && !TOL;  // 1/h and sqrt(g h) staged per cell
    constexpr int NW = NT / 64;
    __shared__ double s_q[4][CH];  // eta, hu, hv, b of the chunk (TOL: h, wu, wv, b)
    // CLEAR: 1/h and sqrt(g h) of each cell (clear_cell); TOL: sqrt(g h) (0 when dry)
    __shared__ double s_x[CLEAR ? 2 : 1][CLEAR || TOL ? CH : 1];
    __shared__ double s_f[4][3][CH];  // flux (h, hu, hv, s) per (edge, cell)
    // The edge list (swe_device.hpp).  RAW meshes are not validated: their
    // leaving edges' neighbours are read again instead of listed.
    __shared__ uint32_t s_list[3 * CH + 4];
    __shared__ uint32_t s_jb[JUMPS ? CH / 16 : 1];  // elevation-jump bits, 2 per cell
    __shared__ int s_wsum[NW];
    __shared__ double s_wmax[NW], s_dt;
    __shared__ int s_wref[NW];
    // geometry tables in LDS: the per-lane indexed reads would otherwise be
    // global loads that every edge waits for
    __shared__ double s_dir[8][2];  // the unit vectors at multiples of 45 degrees
    __shared__ double s_leg[64];

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    // the hypotenuse normals of plotter types 1..8 point to 90, 135, ... degrees
    if (t < 16) s_dir[t >> 1][t & 1] = c_normal[((((t >> 1) - 2) & 7) + 9) * 6 + 2 + (t & 1)];
    for (int i = t; i < 64; i += NT) s_leg[i] = c_leg[i];

    // XCD-aware order: virtual block v runs on XCD v % 8 (the dispatcher deals
    // workgroups round robin and the grid is a multiple of 8); XCD x owns a
    // contiguous range of chunks.
    // (there are fewer than 2^31 chunks)
    const uint32_t nchunks = (uint32_t)args.nchunks, q = nchunks / 8, r = nchunks % 8;
    const uint32_t nvirt = 8 * ((nchunks + 7) / 8);
    for (uint32_t v = blockIdx.x; v < nvirt; v += gridDim.x) {
        const uint32_t xcd = v % 8, i = v / 8;
        if (i >= q + (xcd < r ? 1 : 0)) continue;  // uniform across the workgroup
        const uint32_t chunk = xcd * q + (xcd < r ? xcd : r) + i;
        // The arguments are read where they are used, for each chunk (the
        // empty asm hides that the address is the same every time): held
        // across the loop, they and what is derived from them outgrow the
        // scalar registers, and every wave moved them to vector lanes first.
        auto ap = (const __attribute__((address_space(4))) StepArgs *)
            __builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(ap));
        const auto &a = *ap;
        const double g = a.g, inv16g = a.inv16g;
        // Raised wave priority from here to the edge loop: the chunk's
        // descriptor and staging loads, and the edge list, are a chain of
        // memory round trips and barriers; issued ahead of the other waves'
        // solver arithmetic, they overlap it (3-5 % off the step).
        __builtin_amdgcn_s_setprio(2);
        // What is uniform is read through the scalar cache; one scenario's
        // table entry comes with the arguments, so that its state loads do
        // not wait for a table read.
        const int s = !RAW && a.chunk_scen ? scalar(a.chunk_scen)[chunk] : 0;
        const auto *const sp = !RAW && a.chunk_scen ? scalar(a.scen) + s : &a.scen0;
        const auto &sc = *sp;
        // The state and topology arrays are addressed from per-scenario
        // (gs_*) and per-chunk (c_*) base pointers that are uniform across
        // the workgroup; cell indices are 32-bit (a scenario holds at most
        // 2^29 cells).
        const int32_t lbase = (int32_t)(chunk - (uint32_t)sc.chunk_off) * CH;  // first cell of the chunk
        const int cnt = (int)((sc.n - lbase) < CH ? (sc.n - lbase) : CH);
        const bool active = t < cnt;
        const int64_t gs = sc.cell_off, gt = sc.topo_off;  // state / topology offsets
        const double *const gs_eta = a.eta + gs, *const gs_hu = a.hu + gs, *const gs_hv = a.hv + gs;
        const double *const gs_b = a.b + gs;
        const double *const c_eta = gs_eta + lbase, *const c_hu = gs_hu + lbase;
        const double *const c_hv = gs_hv + lbase, *const c_b = gs_b + lbase;
        const int32_t *const c_nbr = a.nbr + 3 * (gt + lbase);
        const int8_t *const c_plot = a.plotter + gt + lbase;
        const int8_t *const c_depth = a.depth + gt + lbase;
        const uint32_t *const list =
            !RAW && a.lists ? a.lists + (uint64_t)chunk * list_words(CH) : nullptr;
        const int64_t c_out = gs + lbase;  // first output cell of the chunk
        double dt = a.device_dt ? scalar(a.slots)[s].dt
                                : (a.dt_host ? scalar(a.dt_host)[s] : a.dt);
        const double drytol = sc.drytol;

        // a chain: the last step's fastest cell, from its chunks' partials
        // (the minimum waits for the loads only after the staging's)
        double fastest = 0.0;
        if (!RAW && a.prev_max) {
            const int n = a.chunk_scen ? (int)sc.nchunks : a.prev_chunks;
            const double *const pm = a.prev_max + (a.chunk_scen ? sc.chunk_off : 0);
            for (int i0 = t; i0 < n; i0 += NT) fastest = max_f64(fastest, pm[i0]);
        }

        // the stored list, or this thread's cell's neighbours to build it from
        int32_t nb[3] = {-1, -1, -1};
        int plot = 1;
        uint32_t head = 0;
        ListAhead<CH, NT> ahead;
        if (list) {
            head = scalar(list)[0];
            ahead.load(list, t);
        } else if (active) {
            nb[0] = c_nbr[3 * t];
            nb[1] = c_nbr[3 * t + 1];
            nb[2] = c_nbr[3 * t + 2];
            plot = c_plot[t];
        }
        double my_e = 0.0, my_u = 0.0, my_v = 0.0;  // TOL: this thread's cell state
        if (active) {
            // every load goes out before the arithmetic that waits for the state
            const double e = c_eta[t], u = c_hu[t], vv = c_hv[t], bb = c_b[t];
            if constexpr (TOL) {
                my_e = e;
                my_u = u;
                my_v = vv;
                const tol::CellQ cq = tol::cell_q(e, u, vv, bb, drytol, g);
                s_q[0][t] = cq.h;
                s_q[1][t] = cq.wu;
                s_q[2][t] = cq.wv;
                s_q[3][t] = cq.b;
                s_x[0][t] = cq.sq;
            } else {
                s_q[0][t] = e;
                s_q[1][t] = u;
                s_q[2][t] = vv;
                s_q[3][t] = bb;
                if constexpr (CLEAR) {
                    const ClearCell k = clear_cell<SOLVER>(e, u, vv, bb, drytol, g);
                    s_x[0][t] = k.r;
                    s_x[1][t] = k.c;
                }
            }
            if (RAW) {  // a neighbour outside the mesh reads as the boundary
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if ((uint32_t)nb[k] >= (uint64_t)sc.n) nb[k] = -1;
            }
        }
        // RAW: the chunk's neighbours, for the back edges; the flux slots are
        // not written before the edge loop
        int32_t *const s_nbr = reinterpret_cast<int32_t *>(&s_f[0][0][0]);
        if (RAW && t < CH) {
#pragma unroll
            for (int k = 0; k < 3; ++k) s_nbr[k * CH + t] = nb[k];
        }
        if (JUMPS && t < CH / 16) s_jb[t] = 0;

        if (!RAW && a.prev_max) {
            const double w = wave_max(fastest);
            if (lane == 63) s_wmax[wave] = w;
        }
        int2 entries;
        if (list) {
            entries = ahead.put(list, head, t, s_list);
        } else {
            // a plain neighbour's edge back to this cell (two cells of a
            // conforming mesh share at most one edge)
            auto back = [&](int k, int lo) -> int {
                if (!RAW) return nb[k] & 3;
                return s_nbr[lo] == lbase + t ? 0 : (s_nbr[CH + lo] == lbase + t ? 1 : 2);
            };
            auto put = [&](int i, uint32_t ent) { s_list[i] = ent; };
            entries = list_edges<NT, RAW>(t, cnt, lbase, nb, plot, s_wsum, back, put);
        }
        const int n_inner = entries.x, total = entries.y;
        __syncthreads();
        if (!RAW && a.prev_max && t == 0) {
            double m = s_wmax[0];
#pragma unroll
            for (int w = 1; w < NW; ++w) m = max_f64(m, s_wmax[w]);
            s_dt = next_dt(sc.courant, sc.dt_clamp, cfl_minimum(sc.scaling, m));
        }
        // inner edges are solved from their left side: the lower cell when
        // forward, the upper when backward, whose normal is the opposite one
        const int left = a.forward ? 0 : 11, right = 11 - left;
        const uint32_t opposite = a.forward ? 0u : 4u;

        __builtin_amdgcn_s_setprio(0);
        // One pass over the list.  FIRST: a GeoClaw kernel's pass with clear_flux,
        // which leaves the rounds (of NT entries) where one of a wave's edges
        // is not clear to a second pass with the general solver; returns their
        // bits, the same for the whole wave.  A pass of its own keeps the
        // general solver's registers from adding to the shortcut's.
        auto solve = [&](auto first_pass, uint32_t rounds) -> uint32_t {
        constexpr bool FIRST = decltype(first_pass)::value;
        constexpr bool SHORT = GEOCLAW && FIRST;
        uint32_t rest = 0, bit = 1;
        for (int e = t; e < total; e += NT, bit <<= 1) {
            if (!FIRST && !(rounds & bit)) continue;
            const uint32_t ent = s_list[e];
            const bool inside = !(ent & LEAVES);
            const int lc = (ent >> left) & 511, k = (ent >> (left + 9)) & 3;
            const uint32_t dir = ((ent >> 22) & 7) ^ (inside ? opposite : 0u);
            double nx = s_dir[dir][0], ny = s_dir[dir][1];
            // the two cells' quantities: left and right for an inner edge;
            // one that leaves the chunk may need them exchanged
            double L[6] = {}, R[6] = {};
#pragma unroll
            for (int m = 0; m < 4; ++m) L[m] = s_q[m][lc];
            if (SHORT || TOL) L[4] = s_x[0][lc];
            if (SHORT && CLEAR) L[5] = s_x[CLEAR ? 1 : 0][lc];
            const int lo = (ent >> right) & 511;
            bool flip = false;
            uint32_t jb = 0;
            if (inside) {
#pragma unroll
                for (int m = 0; m < 4; ++m) R[m] = s_q[m][lo];
                if (SHORT || TOL) R[4] = s_x[0][lo];
                if (SHORT && CLEAR) R[5] = s_x[CLEAR ? 1 : 0][lo];
            } else if (ent & BOUNDARY) {
                // ghost state of bnd_skeleton_scalar_op (outflow copy or mirror)
#pragma unroll
                for (int m = 0; m < 6; ++m) R[m] = L[m];
                if (a.bc == 1) {
                    const double dp = L[1] * nx + L[2] * ny;
                    R[1] = L[1] - (2.0 * dp) * nx;
                    R[2] = L[2] - (2.0 * dp) * ny;
                }
            } else {
                const int32_t p = RAW ? c_nbr[3 * lc + k] : (int32_t)s_list[e + total - n_inner];
                const int32_t o = RAW ? p : p >> 2;
                R[0] = gs_eta[o];
                R[1] = gs_hu[o];
                R[2] = gs_hv[o];
                R[3] = gs_b[o];
                if constexpr (TOL) {
                    const tol::CellQ cq = tol::cell_q(R[0], R[1], R[2], R[3], drytol, g);
                    R[0] = cq.h;
                    R[1] = cq.wu;
                    R[2] = cq.wv;
                    R[4] = cq.sq;
                }
                if constexpr (SHORT && CLEAR) {
                    const ClearCell x = clear_cell<SOLVER>(R[0], R[1], R[2], R[3], drytol, g);
                    R[4] = x.r;
                    R[5] = x.c;
                }
                flip = a.forward ? o < lbase : o > lbase;  // the other cell comes first
            }
            if constexpr (JUMPS && FIRST) {
                // the elevation jump across an edge between two wet cells:
                // bit 0 if above the refinement tolerance, bit 1 if not below
                // the coarsening tolerance (a NaN jump sets neither); the
                // same for both cells, as |a - b| = |b - a|
                const double hl = TOL ? L[0] : L[0] - L[3], hr = TOL ? R[0] : R[0] - R[3];
                const double jd = TOL ? fabs((L[0] + L[3]) - (R[0] + R[3])) : fabs(L[0] - R[0]);
                if (!(ent & BOUNDARY) && hl > drytol && hr > drytol)
                    jb = (jd > a.jump_refine ? 1u : 0u) | (jd >= a.jump_coarsen ? 2u : 0u);
                if (jb) {
                    atomicOr(&s_jb[lc >> 4], jb << (2 * (lc & 15)));
                    if (inside) atomicOr(&s_jb[lo >> 4], jb << (2 * (lo & 15)));
                }
            }
            const bool flips = __ballot(flip) != 0;  // no wave of inner edges does
            if (flips) {
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    const double x = L[m];
                    L[m] = flip ? R[m] : x;
                    R[m] = flip ? x : R[m];
                }
                nx = flip ? -nx : nx;
                ny = flip ? -ny : ny;
            }
            Flux fL, fR;
            if constexpr (SHORT) {
                // normal and tangential velocities (and momenta) of both sides
                ClearEdge ce;
                const double hL = TOL ? L[0] : L[0] - L[3], hR = TOL ? R[0] : R[0] - R[3];
                const double cL = TOL ? L[4] : L[5], cR = TOL ? R[4] : R[5];
                bool clear;
                if constexpr (TOL) {
                    ce.uL = nx * L[1] + ny * L[2];
                    ce.vL = nx * L[2] - ny * L[1];
                    ce.uR = nx * R[1] + ny * R[2];
                    ce.vR = nx * R[2] - ny * R[1];
                    clear = tol::is_clear<SOLVER>(ce.uL, ce.uR, cL, cR);
                } else {
                    ce = clear_edge(nx, ny, hL, L[1], L[2], L[4], hR, R[1], R[2], R[4]);
                    clear = is_clear<SOLVER>(ce.uL, ce.uR, cL, cR);
                }
                const bool dead = hL <= drytol && hR <= drytol;
                if (__ballot(!dead && !clear) != 0) {
                    rest |= bit;
                    continue;
                }
                if constexpr (TOL)
                    tol::clear_flux<SOLVER>(nx, ny, hL, ce.uL, ce.vL, L[3], cL, hR, ce.uR, ce.vR,
                                            R[3], cR, g, fL, fR);
                else
                    clear_flux<SOLVER>(nx, ny, ce, hL, L[3], cL, hR, R[3], cR, g, fL, fR);
                if (__ballot(dead) != 0 && dead) fL = fR = Flux{0.0, 0.0, 0.0, 0.0};
            } else if constexpr (TOL) {
                tol::edge_flux<SOLVER>(nx, ny, L[0], L[1], L[2], L[3], L[4], R[0], R[1], R[2], R[3],
                                       R[4], drytol, g, inv16g, fL, fR);
            } else {
                edge_flux<SOLVER>(nx, ny, L[0], L[1], L[2], L[3], R[0], R[1], R[2], R[3], drytol, g,
                                  inv16g, fL, fR);
            }
            if (flips && flip) fL = fR;
            s_f[0][k][lc] = fL.h;
            s_f[1][k][lc] = fL.hu;
            s_f[2][k][lc] = fL.hv;
            s_f[3][k][lc] = fL.s;
            if (inside) {
                const int ko = (ent >> (right + 9)) & 3;
                s_f[0][ko][lo] = fR.h;
                s_f[1][ko][lo] = fR.hu;
                s_f[2][ko][lo] = fR.hv;
                s_f[3][ko][lo] = fR.s;
            }
        }
        return rest;
        };
        const uint32_t rest = solve(std::true_type{}, 0u);
        if constexpr (GEOCLAW) {
            if (rest) (void)solve(std::false_type{}, rest);
        }
        __syncthreads();

        // cell update: volume_op + cell_update_op
        if (!RAW && a.prev_max) dt = s_dt;
        if (a.chained && lbase == 0 && t == 0) a.slots[s].time = a.slots[s].time + dt;
        // The CFL candidate of a cell is fl(volume / sv), volume = S^2 2^-(d+1):
        // scaling by a power of two is exact and the rounded quotient falls
        // as the divisor grows, so a mesh's minimum is the quotient of S^2
        // and the largest sv 2^(d+1) (a cell whose sv is NaN has no limit).
        double speed = 0.0;
        bool refined = false;
        if (active) {
            const int d = sc.depth >= 0 ? sc.depth : (int)c_depth[t];
            const double S = sc.scaling;
            const double volume = (S * S) * ldexp(1.0, -(d + 1));
            const double lleg = S * s_leg[d + 1], lhyp = S * s_leg[d];
            const int k0 = a.forward ? 0 : 2, k2 = a.forward ? 2 : 0;
            double dh = 0.0, d1 = 0.0, d2 = 0.0, sv = 0.0;
            dh = dh + lleg * s_f[0][k0][t];
            d1 = d1 + lleg * s_f[1][k0][t];
            d2 = d2 + lleg * s_f[2][k0][t];
            sv = sv + lleg * s_f[3][k0][t];
            dh = dh + lhyp * s_f[0][1][t];
            d1 = d1 + lhyp * s_f[1][1][t];
            d2 = d2 + lhyp * s_f[2][1][t];
            sv = sv + lhyp * s_f[3][1][t];
            dh = dh + lleg * s_f[0][k2][t];
            d1 = d1 + lleg * s_f[1][k2][t];
            d2 = d2 + lleg * s_f[2][k2][t];
            sv = sv + lleg * s_f[3][k2][t];

            int8_t rf = 0;
            if constexpr (JUMPS) {
                // elevation jumps to the wet neighbours of a wet cell, in
                // the state the step reads, from the edge loop's bits: bit 0
                // if one is above the refinement tolerance, bit 1 if one is
                // not below the coarsening tolerance.  j = the largest jump
                // (0 without a wet neighbour): j > tol if some edge's is,
                // j < tol if every edge's is and tol > 0.
                const int jb = (s_jb[t >> 4] >> (2 * (t & 15))) & 3;
                if (d < sc.dmax && (jb & 1)) {
                    rf = 1;
                    refined = true;
                } else if (d > sc.dmin && !(jb & 2) && a.jump_coarsen > 0.0) {
                    rf = -1;
                }
            } else {
                const double dq = fabs(dh);
                if (d < sc.dmax && dq > sc.refine_thr) {
                    rf = 1;
                    refined = true;
                } else if (d > sc.dmin && dq < sc.refine_thr / 8.0) {
                    rf = -1;
                }
            }
            if (a.refine) a.refine[c_out + t] = rf;
            speed = ldexp(sv, d + 1);
            const double scale = -dt / volume;
            dh = scale * dh;
            d1 = scale * d1;
            d2 = scale * d2;

            double qh = TOL ? my_e : s_q[0][t], q1 = TOL ? my_u : s_q[1][t];
            double q2 = TOL ? my_v : s_q[2][t];
            const double qb = s_q[3][t];
            int mk = 0;
            if (qh < qb + drytol && dh > 0.0) {  // wetting, :271-275
                qh = qb + drytol;
                q1 = 0.0;
                q2 = 0.0;
                mk = 1;
            }
            qh = qh + dh;
            q1 = q1 + d1;
            q2 = q2 + d2;
            if (qh < qb + drytol) {  // drying, :280-283
                qh = dmin2(qb, 0.0);
                q1 = 0.0;
                q2 = 0.0;
                mk |= 2;
            }
            if (a.masks) a.masks[c_out + t] = (int8_t)mk;
            a.eta_out[c_out + t] = qh;
            a.hu_out[c_out + t] = q1;
            a.hv_out[c_out + t] = q2;
        }

        // CFL minimum and refinement count of the chunk (post_traversal_grid_op
        // :117-118), reduced over the scenario here, later, or in the next step.
        const double wmax = wave_max(speed);
        const int wref = __popcll(__ballot(refined));
        if (lane == 63) {
            s_wmax[wave] = wmax;
            s_wref[wave] = wref;
        }
        __syncthreads();
        if (t == 0) {
            // from 0: a chunk of NaN sets no limit (meet compares bits, where
            // a NaN is above every number)
            double m = max_f64(0.0, s_wmax[0]);
            int rsum = s_wref[0];
#pragma unroll
            for (int w = 1; w < NW; ++w) {
                m = max_f64(m, s_wmax[w]);
                rsum += s_wref[w];
            }
            if (!RAW && a.meet) {
                long long all = rsum;
                if (meet(a.meet + (int64_t)s * MEET_SLOTS, chunk - (uint32_t)sc.chunk_off,
                         (uint32_t)sc.nchunks, m, all)) {
                    const double c = cfl_minimum(sc.scaling, m);
                    a.slots[s].res_dtcfl = c;
                    a.slots[s].res_nref = all;
                    if (a.out_dtcfl) a.out_dtcfl[s] = c;
                    if (a.out_nref) a.out_nref[s] = all;
                    if (a.device_dt) {
                        a.slots[s].time = a.slots[s].time + dt;
                        a.slots[s].dt = next_dt(sc.courant, sc.dt_clamp, c);
                    }
                }
            } else {
                a.part_max[chunk] = m;
                a.part_nref[chunk] = rsum;
            }
        }
        __syncthreads();  // LDS is reused by the next chunk
    }
}

__global__ __launch_bounds__(FIN_THREADS) void finalize_kernel(StepArgs a) {
    finalize_scenario(a, blockIdx.x);
}

hipError_t upload_tables(const double *normal, const double *leg) {
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_normal), normal, sizeof(double) * 17 * 3 * 2);
    if (e != hipSuccess) return e;
    return hipMemcpyToSymbol(HIP_SYMBOL(c_leg), leg, sizeof(double) * 64);
}

hipError_t launch_finalize(const StepArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(finalize_kernel, dim3((unsigned)a.n_scen), dim3(FIN_THREADS), 0, s, a);
    return hipGetLastError();
}

// The edge list of each chunk: the step kernels' own (list_edges), stored.
template <int CH>
__global__ __launch_bounds__(CH) void edge_list_kernel(StepArgs a, uint32_t *lists) {
    __shared__ int s_wsum[CH / 64];
    const int t = threadIdx.x;
    const uint32_t chunk = blockIdx.x;
    const int s = a.chunk_scen ? a.chunk_scen[chunk] : 0;
    const Scen sc = a.chunk_scen ? a.scen[s] : a.scen0;
    const int32_t lbase = (int32_t)(chunk - (uint32_t)sc.chunk_off) * CH;
    const int cnt = (int)((sc.n - lbase) < CH ? (sc.n - lbase) : CH);
    const int32_t *const nbr = a.nbr + 3 * (sc.topo_off + lbase);
    int32_t nb[3] = {-1, -1, -1};
    int plot = 1;
    if (t < cnt) {
        nb[0] = nbr[3 * t];
        nb[1] = nbr[3 * t + 1];
        nb[2] = nbr[3 * t + 2];
        plot = a.plotter[sc.topo_off + lbase + t];
    }
    uint32_t *const list = lists + (uint64_t)chunk * list_words(CH);
    const int2 n = list_edges<CH, false>(
        t, cnt, lbase, nb, plot, s_wsum, [&](int k, int) { return nb[k] & 3; },
        [&](int i, uint32_t ent) { list[LIST_HEAD + i] = ent; });
    if (t == 0) list[0] = (uint32_t)n.x | ((uint32_t)n.y << 16);
}

size_t edge_list_bytes(int64_t nchunks, int chunk) {
    return sizeof(uint32_t) * (size_t)list_words(chunk) * (size_t)nchunks;
}

hipError_t build_edge_lists(const StepArgs &a, int chunk, uint32_t *lists, hipStream_t s) {
    const dim3 grid((unsigned)a.nchunks);
    switch (chunk) {
        case 128: edge_list_kernel<128><<<grid, 128, 0, s>>>(a, lists); break;
        case 256: edge_list_kernel<256><<<grid, 256, 0, s>>>(a, lists); break;
        case 512: edge_list_kernel<512><<<grid, 512, 0, s>>>(a, lists); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int SOLVER, int CH, int NT>
static void launch_nt(const StepArgs &a, unsigned blocks, hipStream_t s) {
    constexpr bool GEOCLAW = SOLVER == 0 || SOLVER == 1;  // the toleranced solvers
    if (GEOCLAW && a.tol) {
        if (a.flag_jumps)
            hipLaunchKernelGGL((euler_step_kernel<SOLVER, CH, NT, true, false, GEOCLAW>),
                               dim3(blocks), dim3(NT), 0, s, a);
        else
            hipLaunchKernelGGL((euler_step_kernel<SOLVER, CH, NT, false, false, GEOCLAW>),
                               dim3(blocks), dim3(NT), 0, s, a);
    } else if (a.flag_jumps)
        hipLaunchKernelGGL((euler_step_kernel<SOLVER, CH, NT, true>), dim3(blocks), dim3(NT), 0, s,
                           a);
    else
        hipLaunchKernelGGL((euler_step_kernel<SOLVER, CH, NT, false>), dim3(blocks), dim3(NT), 0,
                           s, a);
}

template <int SOLVER, int CH>
static void launch_t(const StepArgs &a, int64_t grid_blocks, hipStream_t s) {
    const int64_t nvirt = 8 * ((a.nchunks + 7) / 8);
    const int64_t blocks = grid_blocks > 0 && grid_blocks < nvirt ? grid_blocks : nvirt;
    // Two threads per cell where every workgroup is resident at once that way
    // (256 CUs of 1024 lanes at this kernel's registers): a chunk's ~1.6 CH
    // edges then take one round instead of two, and the launch is as long as
    // its slowest chunk.  100 steps: 1.38 -> 1.25 ms at 32 chunks, 1.54 ->
    // 1.40 at 256, 1.79 -> 1.72 at 512; 2.42 -> 2.87 at 1024, and a full
    // chip's step 134 -> 200 us.
    if (CH <= 256 && a.nchunks * 2 * CH <= 256 * 1024)
        launch_nt<SOLVER, CH, CH <= 256 ? 2 * CH : CH>(a, (unsigned)blocks, s);
    else
        launch_nt<SOLVER, CH, CH>(a, (unsigned)blocks, s);
    if (!a.skip_finalize && !a.meet)
        hipLaunchKernelGGL(finalize_kernel, dim3((unsigned)a.n_scen), dim3(FIN_THREADS), 0, s, a);
}

template <int SOLVER>
static hipError_t launch_chunk(const StepArgs &a, int chunk, int64_t grid_blocks, hipStream_t s) {
    switch (chunk) {
        case 128: launch_t<SOLVER, 128>(a, grid_blocks, s); break;
        case 256: launch_t<SOLVER, 256>(a, grid_blocks, s); break;
        case 512: launch_t<SOLVER, 512>(a, grid_blocks, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int SOLVER>
static void launch_raw_t(const StepArgs &a, hipStream_t s) {
    constexpr int CH = DEFAULT_CHUNK;
    const int64_t nvirt = 8 * ((a.nchunks + 7) / 8);
    hipLaunchKernelGGL((euler_step_kernel<SOLVER, CH, CH, false, true>), dim3((unsigned)nvirt),
                       dim3(CH), 0, s, a);
    hipLaunchKernelGGL(finalize_kernel, dim3(1), dim3(FIN_THREADS), 0, s, a);
}

hipError_t launch_step_raw(const StepArgs &a, int solver, hipStream_t s) {
    if (a.scen || a.chunk_scen || a.n_scen != 1 || !a.raw_nbr || a.flag_jumps ||
        a.nchunks != (a.scen0.n + DEFAULT_CHUNK - 1) / DEFAULT_CHUNK)
        return hipErrorInvalidValue;
    switch (solver) {
        case 0: launch_raw_t<0>(a, s); break;
        case 1: launch_raw_t<1>(a, s); break;
        case SOLVER_LF: launch_raw_t<SOLVER_LF>(a, s); break;
        case SOLVER_LLF: launch_raw_t<SOLVER_LLF>(a, s); break;
        case SOLVER_LF_BATH: launch_raw_t<SOLVER_LF_BATH>(a, s); break;
        case SOLVER_LLF_BATH: launch_raw_t<SOLVER_LLF_BATH>(a, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_step(const StepArgs &a, int solver, int chunk, int64_t grid_blocks,
                       hipStream_t s) {
    if (a.raw_nbr || !a.scen) return hipErrorInvalidValue;
    if (grid_blocks < 0 || grid_blocks % 8) return hipErrorInvalidValue;
    switch (solver) {
        case 0: return launch_chunk<0>(a, chunk, grid_blocks, s);
        case 1: return launch_chunk<1>(a, chunk, grid_blocks, s);
        case SOLVER_LF: return launch_chunk<SOLVER_LF>(a, chunk, grid_blocks, s);
        case SOLVER_LLF: return launch_chunk<SOLVER_LLF>(a, chunk, grid_blocks, s);
        case SOLVER_LF_BATH: return launch_chunk<SOLVER_LF_BATH>(a, chunk, grid_blocks, s);
        case SOLVER_LLF_BATH: return launch_chunk<SOLVER_LLF_BATH>(a, chunk, grid_blocks, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace swe
