// Floats moved between workgroups as device-coherent accesses (agent-scope
// relaxed atomics: sc1 stores and loads on gfx950), which need no fence.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mb {

__device__ __forceinline__ void store_coherent(float* p, float a, float b) {
  const uint64_t v = (uint64_t)__float_as_uint(a) | ((uint64_t)__float_as_uint(b) << 32);
  __hip_atomic_store((uint64_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load_coherent(const float* p, float& a, float& b) {
  const uint64_t v = __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  a = __uint_as_float((uint32_t)v);
  b = __uint_as_float((uint32_t)(v >> 32));
}
__device__ __forceinline__ float4 load_coherent(const float* p) {
  float4 r;
  load_coherent(p, r.x, r.y);
  load_coherent(p + 2, r.z, r.w);
  return r;
}

}  // namespace mb
