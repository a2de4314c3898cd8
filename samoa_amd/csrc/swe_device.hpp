// swe_device.hpp -- what the step kernel and its adjoint share on the device.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace swe {

// A pointer to memory that no kernel writes while this one runs, for scalar
// loads from uniform addresses.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *scalar(const T *p) {
    return (const __attribute__((address_space(4))) T *)p;
}

// Lanes of the mask below this one.
__device__ __forceinline__ int lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

// A chunk's edge list.  Entries of the edges inside it come first (each once,
// from its lower cell), then those leaving it (to other chunks or the domain
// boundary), then the packed neighbours of the latter.  An entry holds the lower
// cell and its edge (bits 0-10), the upper cell and its edge (bits 11-21) and
// the direction of the lower cell's outward normal in multiples of 45 degrees
// (bits 22-24).  A leaving edge holds its cell twice.
//
// A chunk of m cells of a validated mesh has at least m - 1 inner edges
// (consecutive cells share one), so at most m + 2 leave it: inner + 2 leaving
// = (3 m + 3 leaving) / 2 <= 3 m + 3 entries.
constexpr uint32_t LEAVES = 1u << 31, BOUNDARY = 1u << 30;

// Words of a stored list: inner entries | all entries << 16, three unused, the
// entries.
constexpr int LIST_HEAD = 4;
constexpr int list_words(int chunk) { return LIST_HEAD + 3 * chunk + 4; }

// Builds the list from this thread's cell's neighbours (packed, -1 without one)
// and plotter type; threads t >= cnt have none.  back(k, lo): edge of the
// neighbour lo in the chunk that is this cell's edge k; put(i, entry).  Returns
// inner and all entries, the same for every thread; holds one barrier.
template <int NT, bool RAW, class Back, class Put>
__device__ __forceinline__ int2 list_edges(int t, int cnt, int32_t lbase, const int32_t (&nb)[3],
                                           int plot, int *s_wsum, Back back, Put put) {
    const int lane = t & 63, wave = t >> 6;
    int inner = 0, leave = 0;
    if (t < cnt) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int32_t p = nb[k];
            const int lo = (RAW ? p : p >> 2) - lbase;  // chunk-local neighbour
            const bool inside = p >= 0 && (uint32_t)lo < (uint32_t)cnt;
            if (!inside) leave |= 1 << k;
            else if (lo > t) inner |= 1 << k;
        }
    }
    // workgroup exclusive prefixes of both counts (0..3 each) via ballots,
    // packed: inner in the low half, leaving in the high half
    const int nin = __popc(inner), nout = __popc(leave);
    const uint64_t i0 = __ballot(nin & 1), i1 = __ballot(nin & 2);
    const uint64_t o0 = __ballot(nout & 1), o1 = __ballot(nout & 2);
    const int wpre = lanes_below(i0) + 2 * lanes_below(i1) +
                     ((lanes_below(o0) + 2 * lanes_below(o1)) << 16);
    if (lane == 0)
        s_wsum[wave] = __popcll(i0) + 2 * __popcll(i1) +
                       ((__popcll(o0) + 2 * __popcll(o1)) << 16);
    __syncthreads();
    int pre = wpre, sum = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        const int ws = s_wsum[w];
        pre += w < wave ? ws : 0;
        sum += ws;
    }
    const int n_inner = sum & 0xffff, total = n_inner + (sum >> 16);
    int pi = pre & 0xffff, po = n_inner + (pre >> 16);
    // outward normal of edge k: plotter type p > 0 turns the normals at
    // 180 + 45 p, 45 + 45 p and 270 + 45 p degrees, p < 0 mirrors the legs
    const int turn = plot < 0 ? -plot : plot;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int d0 = k == 1 ? 1 : ((k == 0) == (plot > 0) ? 4 : 6);
        const int32_t p = nb[k];
        const bool in = inner & (1 << k), out = leave & (1 << k);
        const uint32_t self = (uint32_t)t | ((uint32_t)k << 9);
        const int lo = (RAW ? p : p >> 2) - lbase;
        const uint32_t other =
            in ? ((uint32_t)lo << 11) | ((uint32_t)back(k, lo) << 20)
               : (self << 11) | LEAVES | (p < 0 ? BOUNDARY : 0u);
        if (in || out) put(in ? pi : po, self | ((uint32_t)((turn + d0) & 7) << 22) | other);
        if (!RAW && out) put(po + total - n_inner, (uint32_t)p);
        pi += in ? 1 : 0;
        po += out ? 1 : 0;
    }
    return make_int2(n_inner, total);
}

// This workgroup's part of a stored list's first words, read ahead of the
// header (they lie inside the list, whatever it holds): the chunk's loads
// wait for memory once.
template <int CH, int NT>
struct ListAhead {
    static constexpr int N = 2 * CH / NT;
    static_assert(N == 1 || N == 2, "one or two threads per cell");
    uint32_t e[N];
    __device__ __forceinline__ void load(const uint32_t *list, int t) {
#pragma unroll
        for (int j = 0; j < N; ++j) e[j] = list[LIST_HEAD + j * NT + t];
    }
    // puts the list into LDS; returns inner and all entries
    __device__ __forceinline__ int2 put(const uint32_t *list, uint32_t head, int t,
                                        uint32_t *s_list) const {
        const int n_inner = (int)(head & 0xffffu), total = (int)(head >> 16);
#pragma unroll
        for (int j = 0; j < N; ++j) s_list[j * NT + t] = e[j];
        for (int i = N * NT + t; i < 2 * total - n_inner; i += NT) s_list[i] = list[LIST_HEAD + i];
        return make_int2(n_inner, total);
    }
};

}  // namespace swe
