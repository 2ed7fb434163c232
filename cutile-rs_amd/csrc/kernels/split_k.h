// One output block computed by several workgroups that share K.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_common.h"

namespace cutile {
namespace gemm {

// ---- partial sums of one output block computed by several workgroups (split K) -----------------------------------------
// The launch's workspace holds, per output block, one f32 copy of the block per K split and a counter that is 0 between
// launches.  The splits of a block run on different XCDs, whose L2 caches are not coherent with each other, so partials
// and counter move with agent-scope accesses (past the L2); the workgroup that counts last adds the partials in split
// order, whatever order they arrived in, so the sum does not depend on timing.
__device__ __forceinline__ void store_partial(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float load_partial(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// eight neighbours at once (8-byte aligned)
__device__ __forceinline__ void store_partials(float* p, const float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p) + i,
                       (uint64_t)__builtin_bit_cast(uint32_t, f[2 * i]) | (uint64_t)__builtin_bit_cast(uint32_t, f[2 * i + 1]) << 32, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load_partials(const float* p, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p) + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    f[2 * i] = __builtin_bit_cast(float, (uint32_t)v);
    f[2 * i + 1] = __builtin_bit_cast(float, (uint32_t)(v >> 32));
  }
}
// Called by the whole workgroup after its partials are stored: true in the workgroup that arrives last of `splits`.
__device__ __forceinline__ bool last_to_arrive(uint32_t* counter, uint32_t splits, uint32_t* shared_flag) {
  __builtin_amdgcn_s_waitcnt(0);   // this wavefront's partials have reached memory
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before == splits - 1) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
    *shared_flag = before == splits - 1;
  }
  __syncthreads();
  return *shared_flag != 0;
}

}  // namespace gemm
}  // namespace cutile
