// swe_adjoint_step.hip -- discrete adjoint of one Euler traversal.
//
// For a traversal Q^{n+1} = F(Q^n, b; dt_n) (swe_step.hip), given the
// adjoint lam^{n+1} = dL/dQ^{n+1}, this kernel computes
//   lam^n  = (dF/dQ^n)^T lam^{n+1}        (eta, hu, hv)
//   gb    += (dF/db)^T   lam^{n+1}
// with dt_n frozen (taken from the forward pass) and the wet/dry limiter
// masks of the forward traversal frozen (cell_update_op,
// SWE_euler_timestep.f90:271-283: bit 0 = wetting fix taken, bit 1 = drying
// fix taken).
//
// Transpose update: the limiter passes the adjoint through, or stops it
// where a fix overwrote a value; the flux sum dQ = s * sum_k len_k f_k
// (s = -dt / vol) then seeds every edge flux of the cell with s * len_k * lam.
// Transpose flux: each edge of the chunk's compacted edge list (the forward
// kernel's, stored with the mesh or built here) runs edge_flux_adj with the seeds
// of both cells, and the gradients with respect to both states are written to
// per-(cell, edge) LDS slots, summed per cell in a fixed order (so results do
// not depend on scheduling).  Edges to cells of other chunks are solved by
// both chunks, each keeping its own side.
//
// What bounds it: FP64 vector issue.  Most edges are clearly subcritical: they
// take clear_flux_adj (660 vector instructions with staging and scatter, the
// same results), the others are compacted into a second list for
// edge_flux_adj (about 1700).  On the d20 tsunami (2.1 M cells) this took the
// kernel from 2740 to 1250 vector instructions per 64 cells, a beach's (d18, a
// fifth of it dry) from 61 to 35 us.  The general pass alone needs 206
// registers: held to 168 it spills 76 bytes on its few edges, and three waves
// per SIMD instead of two hide more of the first pass's LDS and memory waits:
// 213.7 us with neither, 122 with two waves, 106 with three.  LDS (50 KB for
// 256 cells) allows no fourth.  The f-wave kernel went from 107 to 81 us.  A mesh
// of nothing but general edges pays for the first pass: 79 -> 92 us at 524 k cells
// (f-wave 36 -> 42).
//
// Meshes that do not fill the chip are as long as their slowest chunk, and take
// one pass (launch_adj_t): a wave with a general edge solves all of its edges
// so, and there is neither a second list nor a barrier between the passes.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "swe_adjoint.hpp"
#include "swe_adjoint_clear.hpp"
#include "swe_device.hpp"
#include "swe_internal.hpp"

namespace swe {

// Geometry tables of this translation unit (uploaded with the forward ones).
__constant__ double c_normal_adj[17 * 3 * 2];  // [plotter + 8][edge][x,y]
__constant__ double c_leg_adj[64];             // l(k) = sqrt(0.5)**k at k + 1

// NT threads work on a chunk, CH or 2 CH; the first CH hold a cell each.  512 of
// them fill two waves per SIMD, as does the LDS of 512 cells.  ONE: a single
// pass over the list, with the general solver's registers.
template <int SOLVER, int CH, int NT, bool ONE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(ONE || NT == 512 ? 2 : 3))) void
adjoint_step_kernel(AdjArgs args) {
    __shared__ double s_q[4][CH];     // eta, hu, hv, b of the chunk at t_n
    __shared__ double s_x[2][CH];     // 1/h and sqrt(g h) of each cell (clear_cell)
    __shared__ double s_seed[3][CH];  // s * lam^{n+1} after the limiter (per cell)
    __shared__ double s_gb[CH];       // each cell's b gradient so far
    __shared__ double s_g[4][3][CH];  // transpose-flux contributions per (edge, cell)
    __shared__ uint32_t s_list[3 * CH + 4];  // the edge list (swe_device.hpp)
    __shared__ uint16_t s_rest[ONE ? 1 : 3 * CH];  // entries left to the general solver
    __shared__ int8_t s_dep[CH], s_mask[CH];
    __shared__ int s_wsum[NT / 64], s_nrest;
    __shared__ double s_dir[8][2];  // the unit vectors at multiples of 45 degrees
    __shared__ double s_leg[64];

    int t = threadIdx.x;
    if (t < 16) s_dir[t >> 1][t & 1] = c_normal_adj[((((t >> 1) - 2) & 7) + 9) * 6 + 2 + (t & 1)];
    for (int i = t; i < 64; i += NT) s_leg[i] = c_leg_adj[i];
    const uint32_t nchunks = (uint32_t)args.nchunks, q = nchunks / 8, r = nchunks % 8;
    const uint32_t nvirt = 8 * ((nchunks + 7) / 8);
    for (uint32_t v = blockIdx.x; v < nvirt; v += gridDim.x) {
        const uint32_t xcd = v % 8, i = v / 8;
        if (i >= q + (xcd < r ? 1 : 0)) continue;
        const uint32_t chunk = xcd * q + (xcd < r ? xcd : r) + i;
        // read where they are used, for each chunk (see the step kernel)
        auto ap = (const __attribute__((address_space(4))) AdjArgs *)
            __builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(ap));
        const auto &a = *ap;
        // and what follows from t is computed where it is used: LDS addresses
        // kept across the loops are registers that the general solver lacks
        asm volatile("" : "+v"(t));
        // raised wave priority for the chunk's loads and edge list, as in the
        // forward step kernel
        __builtin_amdgcn_s_setprio(2);
        const int s = a.chunk_scen ? scalar(a.chunk_scen)[chunk] : 0;
        const auto &sc = *(scalar(a.scen) + s);
        const int32_t lbase = (int32_t)(chunk - (uint32_t)sc.chunk_off) * CH;
        const int cnt = (int)((sc.n - lbase) < CH ? (sc.n - lbase) : CH);
        const bool active = t < cnt;
        const int64_t gs = sc.cell_off, gt = sc.topo_off;
        const double g = a.g, drytol = sc.drytol, S = sc.scaling;
        const double dt = a.dt_dev ? scalar(a.dt_dev)[s] : a.dt;

        const uint32_t *const list =
            a.lists ? a.lists + (uint64_t)chunk * list_words(CH) : nullptr;

        // the stored list, or this thread's cell's neighbours to build it from
        int32_t nb[3] = {-1, -1, -1};
        int plot = 1;
        uint32_t head = 0;
        ListAhead<CH, NT> ahead;
        if (list) {
            head = scalar(list)[0];
            ahead.load(list, t);
        } else if (active) {
            const int32_t *const nbr = a.nbr + 3 * (gt + lbase);
            nb[0] = nbr[3 * t];
            nb[1] = nbr[3 * t + 1];
            nb[2] = nbr[3 * t + 2];
            plot = a.plotter[gt + lbase + t];
        }
        // transpose of the cell update for this thread's cell
        if (active) {
            // every load in one round: the state, topology, masks and
            // adjoint inputs first, the depth (behind a branch) last
            const int64_t x = gs + lbase + t;
            const double qe = a.eta[x], qu = a.hu[x], qv = a.hv[x], qb = a.b[x];
            const int mk = a.masks[x];
            const double le = a.leta[x], lu = a.lhu[x], lv = a.lhv[x];
            // only this cell's thread adds to its b gradient: read now, with
            // the other loads, not after the edge loop
            s_gb[t] = a.gb[x];
            const int dep = sc.depth >= 0 ? sc.depth : (int)a.depth[gt + lbase + t];
            s_dep[t] = (int8_t)dep;
            s_q[0][t] = qe;
            s_q[1][t] = qu;
            s_q[2][t] = qv;
            s_q[3][t] = qb;
            const ClearCell cc = clear_cell<SOLVER>(qe, qu, qv, qb, drytol, g);
            s_x[0][t] = cc.r;
            s_x[1][t] = cc.c;
            s_mask[t] = (int8_t)mk;
            const bool dry = (mk & 2) != 0;  // drying fix: eta = min(b, 0), p = 0
            const double vol = (S * S) * ldexp(1.0, -(dep + 1));
            const double scale = -dt / vol;
            s_seed[0][t] = scale * (dry ? 0.0 : le);
            s_seed[1][t] = scale * (dry ? 0.0 : lu);
            s_seed[2][t] = scale * (dry ? 0.0 : lv);
        }
        if (t == 0) s_nrest = 0;

        const int2 entries =
            list ? ahead.put(list, head, t, s_list)
                 : list_edges<NT, false>(
                       t, cnt, lbase, nb, plot, s_wsum, [&](int k, int) { return nb[k] & 3; },
                       [&](int i, uint32_t ent) { s_list[i] = ent; });
        const int n_inner = entries.x, total = entries.y;
        __syncthreads();
        // inner edges from their left side, as in the step kernel
        const int left = a.forward ? 0 : 11, right = 11 - left;
        const uint32_t opposite = a.forward ? 0u : 4u;

        __builtin_amdgcn_s_setprio(0);
        // One pass over the list (FIRST, clear_flux_adj; it lists the edges
        // that are not clear, or solves them if it is the only one) or over
        // the rest (edge_flux_adj).  An edge's
        // pass depends on its two states alone and each writes its own
        // slots, so results depend neither on the chunking nor on the order
        // of the rest.  Two passes: the general solver's registers do not
        // add to the shortcut's.
        auto solve = [&](auto first_pass, int n) {
        constexpr bool FIRST = decltype(first_pass)::value;
        asm volatile("" : "+v"(t), "+s"(ap));
        const auto &a = *ap;
        const double g = a.g;
        for (int i = t; i < n; i += NT) {
            const int e = FIRST ? i : s_rest[i];
            const uint32_t ent = s_list[e];
            const bool inside = !(ent & LEAVES);
            const int lc = (ent >> left) & 511, k = (ent >> (left + 9)) & 3;
            const uint32_t dir = ((ent >> 22) & 7) ^ (inside ? opposite : 0u);
            double nx = s_dir[dir][0], ny = s_dir[dir][1];
            // both cells' state, 1/h and c, and seeds: left and right for an
            // inner edge; one that leaves the chunk may need them exchanged
            double L[6] = {}, R[6] = {}, fL[3], fR[3] = {0.0, 0.0, 0.0};
            const int dc = s_dep[lc];
            const double len = S * s_leg[k == 1 ? dc : dc + 1];
#pragma unroll
            for (int m = 0; m < 4; ++m) L[m] = s_q[m][lc];
            if (FIRST) {
                L[4] = s_x[0][lc];
                L[5] = s_x[1][lc];
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) fL[m] = s_seed[m][lc] * len;
            const int lo = (ent >> right) & 511, ko = (ent >> (right + 9)) & 3;
            bool flip = false;
            if (inside) {
#pragma unroll
                for (int m = 0; m < 4; ++m) R[m] = s_q[m][lo];
                if (FIRST) {
                    R[4] = s_x[0][lo];
                    R[5] = s_x[1][lo];
                }
                const int dl = s_dep[lo];
                const double len_o = S * s_leg[ko == 1 ? dl : dl + 1];
#pragma unroll
                for (int m = 0; m < 3; ++m) fR[m] = s_seed[m][lo] * len_o;
            } else if (ent & BOUNDARY) {
#pragma unroll
                for (int m = 0; m < 6; ++m) R[m] = L[m];
                if (a.bc == 1) {
                    const double dp = L[1] * nx + L[2] * ny;
                    R[1] = L[1] - (2.0 * dp) * nx;
                    R[2] = L[2] - (2.0 * dp) * ny;
                }
            } else {
                const int32_t p = (int32_t)s_list[e + total - n_inner], o = p >> 2;
                const int64_t x = gs + o;
                R[0] = a.eta[x];
                R[1] = a.hu[x];
                R[2] = a.hv[x];
                R[3] = a.b[x];
                const int mk = a.masks[x];
                // read with the rest, then selected (a read under the mask
                // test would wait for the mask first)
                const double l0 = a.leta[x], l1 = a.lhu[x], l2 = a.lhv[x];
                const int dl = sc.depth >= 0 ? sc.depth : a.depth[gt + o];
                if (FIRST) {
                    const ClearCell y = clear_cell<SOLVER>(R[0], R[1], R[2], R[3], drytol, g);
                    R[4] = y.r;
                    R[5] = y.c;
                }
                // the neighbour's seed exactly as its own chunk forms it
                // ((s * lam) after the limiter, times the edge length), so
                // that results do not depend on the chunking
                const double vol = (S * S) * ldexp(1.0, -(dl + 1));
                const double scale = -dt / vol;
                const double len_o = S * s_leg[(p & 3) == 1 ? dl : dl + 1];
                const bool dry = (mk & 2) != 0;
                fR[0] = (scale * (dry ? 0.0 : l0)) * len_o;
                fR[1] = (scale * (dry ? 0.0 : l1)) * len_o;
                fR[2] = (scale * (dry ? 0.0 : l2)) * len_o;
                flip = a.forward ? o < lbase : o > lbase;  // the other cell comes first
            }
            const bool flips = __ballot(flip) != 0;  // no wave of inner edges does
            if (flips) {
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    const double x = L[m];
                    L[m] = flip ? R[m] : x;
                    R[m] = flip ? x : R[m];
                }
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                    const double x = fL[m];
                    fL[m] = flip ? fR[m] : x;
                    fR[m] = flip ? x : fR[m];
                }
                nx = flip ? -nx : nx;
                ny = flip ? -ny : ny;
            }
            double gL[4] = {0.0, 0.0, 0.0, 0.0}, gR[4] = {0.0, 0.0, 0.0, 0.0};
            if constexpr (FIRST) {
                const double hL = L[0] - L[3], hR = R[0] - R[3];
                const ClearEdge ce = clear_edge(nx, ny, hL, L[1], L[2], L[4], hR, R[1], R[2], R[4]);
                if constexpr (ONE) {
                    // a wave with a general edge solves all of its edges so
                    const bool clear = is_clear<SOLVER>(ce.uL, ce.uR, L[5], R[5]);
                    bool general =
                        __ballot(!clear && !(hL <= drytol && hR <= drytol)) != 0;
                    if (clear && !general)
                        general = !clear_flux_adj<SOLVER, true>(nx, ny, ce, hL, L[3], L[4], L[5],
                                                                hR, R[3], R[4], R[5], g, fL, fR,
                                                                gL, gR);
                    if (general)
                        edge_flux_adj<SOLVER>(nx, ny, L[0], L[1], L[2], L[3], R[0], R[1], R[2],
                                              R[3], drytol, g, a.inv16g, fL, fR, gL, gR);
                } else if (is_clear<SOLVER>(ce.uL, ce.uR, L[5], R[5])) {
                    if (!clear_flux_adj<SOLVER>(nx, ny, ce, hL, L[3], L[4], L[5], hR, R[3], R[4],
                                                R[5], g, fL, fR, gL, gR)) {
                        s_rest[atomicAdd(&s_nrest, 1)] = (uint16_t)e;
                        continue;
                    }
                } else if (!(hL <= drytol && hR <= drytol)) {
                    s_rest[atomicAdd(&s_nrest, 1)] = (uint16_t)e;
                    continue;
                }
            } else {
                edge_flux_adj<SOLVER>(nx, ny, L[0], L[1], L[2], L[3], R[0], R[1], R[2], R[3], drytol,
                                      g, a.inv16g, fL, fR, gL, gR);
            }
            if (flips) {
#pragma unroll
                for (int m = 0; m < 4; ++m) gL[m] = flip ? gR[m] : gL[m];
            }
            if (ent & BOUNDARY) {  // the ghost is a function of this cell's state
                gL[0] += gR[0];
                gL[3] += gR[3];
                if (a.bc == 1) {
                    const double gdp = -2.0 * (gR[1] * nx + gR[2] * ny);
                    gL[1] += gR[1] + gdp * nx;
                    gL[2] += gR[2] + gdp * ny;
                } else {
                    gL[1] += gR[1];
                    gL[2] += gR[2];
                }
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) s_g[m][k][lc] = gL[m];
            if (inside) {
#pragma unroll
                for (int m = 0; m < 4; ++m) s_g[m][ko][lo] = gR[m];
            }
        }
        };
        solve(std::true_type{}, total);
        __syncthreads();
        if constexpr (!ONE) {
            const int nrest = s_nrest;
            if (nrest) {
                solve(std::false_type{}, nrest);
                __syncthreads();
            }
        }

        asm volatile("" : "+v"(t));
        if (t < cnt) {
            const int64_t x = gs + lbase + t;
            // the limiter's own part, from a second read of the adjoint (in
            // registers across the edge loop it costs a wave per SIMD)
            const int mk = s_mask[t];
            double le = a.leta[x], lu = a.lhu[x], lv = a.lhv[x], lb = 0.0;
            if (mk & 2) {  // drying fix: eta = min(b, 0), p = 0
                if (s_q[3][t] < 0.0) lb += le;
                le = lu = lv = 0.0;
            }
            if (mk & 1) {  // wetting fix: eta = b + drytol, p = 0 before the update
                lb += le;
                le = lu = lv = 0.0;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                le += s_g[0][k][t];
                lu += s_g[1][k][t];
                lv += s_g[2][k][t];
                lb += s_g[3][k][t];
            }
            a.leta_out[x] = le;
            a.lhu_out[x] = lu;
            a.lhv_out[x] = lv;
            a.gb[x] = s_gb[t] + lb;
        }
        __syncthreads();  // LDS is reused by the next chunk
    }
}

hipError_t upload_tables_adjoint(const double *normal, const double *leg) {
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_normal_adj), normal, sizeof(double) * 17 * 3 * 2);
    if (e != hipSuccess) return e;
    return hipMemcpyToSymbol(HIP_SYMBOL(c_leg_adj), leg, sizeof(double) * 64);
}

template <int SOLVER, int CH>
static void launch_adj_t(const AdjArgs &a, int64_t grid_blocks, hipStream_t s) {
    const int64_t nvirt = 8 * ((a.nchunks + 7) / 8);
    const int64_t blocks = grid_blocks > 0 && grid_blocks < nvirt ? grid_blocks : nvirt;
    // Two threads per cell where every workgroup is resident at once that way (256
    // CUs of 512 lanes): a chunk's ~1.6 CH edges then take one round, and the
    // general solver keeps its 205 registers.  A launch of the augmented solver,
    // us: 13.8 -> 11.9 at 8 chunks, 15.0 -> 12.8 at 256, with 128-cell chunks
    // 16.9 -> 14.6 at 512; but 17.4 -> 20.9 at 512 chunks, 24.2 -> 31.7 at 1024.
    //
    // One pass where all are resident (two waves per SIMD) and the launch is as
    // long as a chunk that would pay both: us a launch on a beach (a third of its
    // edges general) with two passes / with one,
    //     f-wave, 256-cell chunks: 1: 6.1 / 4.8, 32: 8.0 / 6.9, 128: 8.2 / 7.0,
    //       256: 8.1 / 7.1, 512: 10.5 / 9.9; every edge general 9.8 / 6.9 at 32,
    //       15.3 / 12.0 at 512; none 5.3 / 5.2 and 8.2 / 8.1
    //     augmented: 1: 10.0 / 8.5, 512: 18.1 / 17.2 (every edge 30.8 / 23.8); with
    //       128-cell chunks 128: 12.7 / 10.8, 512: 16.6 / 12.6
    // With two threads per cell of 256-cell chunks the augmented solver's long
    // branches tell, which a wave in one pass takes for its clear edges too: 12.1 /
    // 13.9 at 4 chunks, 12.3 / 13.9 at 128, 12.9 / 12.8 at 256, and 512-cell chunks
    // 15.6 / 14.1 to 15.7 / 22.3: two passes there.
    constexpr int TWO = CH <= 256 ? 2 * CH : CH;
    constexpr bool SHORT = SOLVER == 1 || CH == 128;
    const int64_t resident = 256 * 512;
    const dim3 grid((unsigned)blocks);
    auto launch = [&](auto threads, auto one) {
        constexpr int NT = decltype(threads)::value;
        constexpr bool ONE = decltype(one)::value;
        hipLaunchKernelGGL((adjoint_step_kernel<SOLVER, CH, NT, ONE>), grid, dim3(NT), 0, s, a);
    };
    using two_threads = std::integral_constant<int, TWO>;
    using one_thread = std::integral_constant<int, CH>;
    if constexpr (CH <= 256) {
        if (a.nchunks * TWO <= resident) {
            if (SHORT || a.nchunks == 1) return launch(two_threads{}, std::true_type{});
            if constexpr (!SHORT) return launch(two_threads{}, std::false_type{});
        }
    }
    if constexpr (SHORT || CH == 256) {
        if (a.nchunks * CH <= resident) return launch(one_thread{}, std::true_type{});
    }
    launch(one_thread{}, std::false_type{});
}

hipError_t launch_adjoint(const AdjArgs &a, int solver, int chunk, int64_t grid_blocks,
                          hipStream_t s) {
    if (grid_blocks < 0 || grid_blocks % 8) return hipErrorInvalidValue;
    if (solver != 0 && solver != 1) return hipErrorInvalidValue;  // the GeoClaw solvers only
    switch (chunk * 2 + (solver == 1 ? 1 : 0)) {
        case 128 * 2: launch_adj_t<0, 128>(a, grid_blocks, s); break;
        case 128 * 2 + 1: launch_adj_t<1, 128>(a, grid_blocks, s); break;
        case 256 * 2: launch_adj_t<0, 256>(a, grid_blocks, s); break;
        case 256 * 2 + 1: launch_adj_t<1, 256>(a, grid_blocks, s); break;
        case 512 * 2: launch_adj_t<0, 512>(a, grid_blocks, s); break;
        case 512 * 2 + 1: launch_adj_t<1, 512>(a, grid_blocks, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace swe
