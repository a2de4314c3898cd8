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

// Flags of the edge list's entries: the edge leaves the chunk, to the domain
// boundary.
constexpr uint32_t LEAVES = 1u << 31, BOUNDARY = 1u << 30;

}  // namespace swe
