// brt_wave.hpp -- lanes of one wave: LDS hand-overs and the four lanes of a quad.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace brt {

// What every lane of the wave wrote to LDS is seen by the others.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The quad's lane K's value; every lane of the quad is active.
template <int K>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, K * 0x55, 0xF, 0xF, true);
}
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
    return __uint_as_float(quad_lane<K>(__float_as_uint(v)));
}

// s + the quad's terms, lane 0's first
__device__ __forceinline__ float quad_add(float s, float v) {
    return (((s + quad_lane<0>(v)) + quad_lane<1>(v)) + quad_lane<2>(v)) + quad_lane<3>(v);
}

}  // namespace brt
