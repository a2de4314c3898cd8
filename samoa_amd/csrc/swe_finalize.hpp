// swe_finalize.hpp -- the reduction of a step's partials and the dt chain.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "swe_internal.hpp"
#include "swe_riemann.hpp"

namespace swe {

// v_max_f64 without the quieting of signalling NaN that fmax adds.
__device__ __forceinline__ double max_f64(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Lane 63 gets the maximum over the wave of values >= 0: row shifts by 1, 2, 4
// and 8, then the rows' last lanes broadcast to the next row and half; a lane
// without a source reads 0.  NaN values are left out, but of 64 of them lane 63
// gets a NaN.
__device__ __forceinline__ double wave_max(double v) {
    auto step = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        v = max_f64(v, __hiloint2double(
                           __builtin_amdgcn_update_dpp(0, __double2hiint(v), C, 0xf, 0xf, true),
                           __builtin_amdgcn_update_dpp(0, __double2loint(v), C, 0xf, 0xf, true)));
    };
    step(std::integral_constant<int, 0x111>{});
    step(std::integral_constant<int, 0x112>{});
    step(std::integral_constant<int, 0x114>{});
    step(std::integral_constant<int, 0x118>{});
    step(std::integral_constant<int, 0x142>{});
    step(std::integral_constant<int, 0x143>{});
    return v;
}

// The CFL minimum (huge(1.0_SR) without a limit, pre_traversal_op :139) from
// the largest sv 2^(d+1), and the dt it gives (post_traversal_grid_op
// :117-118, pre_traversal_grid_op :93-99).
__device__ __forceinline__ double cfl_minimum(double scaling, double fastest) {
    return dmin2(1.7976931348623157e308, (scaling * scaling) / fastest);
}
__device__ __forceinline__ double next_dt(double courant, double dt_clamp, double dt_cfl) {
    const double next = courant * dt_cfl;
    return dt_clamp > 0.0 ? dmin2(dt_clamp, next) : next;
}

constexpr int FIN_THREADS = 1024;

// One workgroup reduces the chunk partials of a scenario's last step, publishes
// the results and advances the device dt chain (post_traversal_grid_op :115-128
// and the next pre_traversal_grid_op :93-99).  Each thread reads FIN_PER partials
// of each array at once (every load at an index in range, the ones past the end
// unused), and the slot's time and dt are read at the start, so that the
// chain of memory round trips is short for meshes up to FIN_PER * FIN_THREADS
// chunks.
constexpr int FIN_PER = 16;
__device__ __forceinline__ void finalize_scenario(const StepArgs &a, int s) {
    __shared__ double s_max[FIN_THREADS / 64];
    __shared__ long long s_ref[FIN_THREADS / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const Scen sc = a.scen ? a.scen[s] : a.scen0;
    Slots *sl = &a.slots[s];
    const double time0 = sl->time, dt0 = sl->dt;  // every thread: no branch to wait at
    double m = 0.0;
    long long r = 0;
    const double *pm = a.part_max + sc.chunk_off;
    const int32_t *pr = a.part_nref + sc.chunk_off;
    // the chunks of the chain's last step, if a remeshing came after it
    const int64_t nc = a.chained && a.n_scen == 1 ? a.prev_chunks : sc.nchunks;
    for (int64_t i0 = t; i0 < nc; i0 += (int64_t)FIN_PER * FIN_THREADS) {
        double v[FIN_PER];
        int32_t w[FIN_PER];
#pragma unroll
        for (int j = 0; j < FIN_PER; ++j) {
            const int64_t i = i0 + (int64_t)j * FIN_THREADS;
            const int64_t ii = i < nc ? i : i0;
            v[j] = pm[ii];
            w[j] = pr[ii];
        }
#pragma unroll
        for (int j = 0; j < FIN_PER; ++j) {
            const bool in = i0 + (int64_t)j * FIN_THREADS < nc;
            m = max_f64(m, in ? v[j] : 0.0);
            r += in ? w[j] : 0;
        }
    }
    m = wave_max(m);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) r += __shfl_xor(r, off, 64);
    if (lane == 63) {
        s_max[wave] = m;
        s_ref[wave] = r;
    }
    __syncthreads();
    if (t == 0) {
        m = s_max[0];
        r = s_ref[0];
#pragma unroll
        for (int w = 1; w < FIN_THREADS / 64; ++w) {
            m = max_f64(m, s_max[w]);
            r += s_ref[w];
        }
        m = cfl_minimum(sc.scaling, m);
        sl->res_dtcfl = m;
        sl->res_nref = r;
        if (a.out_dtcfl) a.out_dtcfl[s] = m;
        if (a.out_nref) a.out_nref[s] = (int64_t)r;
        if (a.device_dt) {
            if (!a.chained) sl->time = time0 + dt0;
            sl->dt = next_dt(sc.courant, sc.dt_clamp, m);
        }
    }
}

}  // namespace swe
