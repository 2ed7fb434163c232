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

// A tile held in a workgroup's accumulators, computed by `splits` workgroups: false in all but the one that arrives last, whose
// accumulators then hold the sum (in split order).  `mine` = the tile's share of the workspace; a partial tile lies there register
// by register, thread by thread: 16 bytes a lane, whole lines, and a thread reads only what its namesakes wrote.
constexpr int kAgentScope = 16;   // buffer accesses with sc1: past the L2, which the XCDs do not share
template <int TM, int TN, int THREADS>
__device__ __forceinline__ bool combine_tile(f32x4 (&acc)[TN][TM], float* mine, uint32_t* counter, uint32_t split, uint32_t splits, uint32_t* shared_flag) {
  constexpr uint32_t kTile = TM * TN * THREADS * 16;   // bytes
  const __amdgpu_buffer_rsrc_t part = make_rsrc(mine, kTile * splits);
#pragma unroll
  for (int r = 0; r < TM * TN; ++r)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[r % TN][r / TN]), part, threadIdx.x * 16, split * kTile + r * (THREADS * 16), kAgentScope);
  if (!last_to_arrive(counter, splits, shared_flag)) return false;
  auto add = [&](uint32_t k) {
#pragma unroll
    for (int r = 0; r < TM * TN; ++r)
      acc[r % TN][r / TN] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(part, threadIdx.x * 16, k * kTile + r * (THREADS * 16), kAgentScope));
  };
  if (splits == 2) {   // a sum of two: either order
    add(1 - split);
    return true;
  }
#pragma unroll
  for (int r = 0; r < TM * TN; ++r) acc[r % TN][r / TN] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t k = 0; k < splits; ++k) add(k);
  return true;
}

// Tile, split and the operands of a launch of tiles_m x tiles_n x splits workgroups (split-major: an XCD's contiguous share is neighbouring
// tiles of one range of K): x, y and k are cut to the K tiles of the split.
struct SplitTile {
  uint32_t pm, pn, tile, split;
};
template <int BK, int BYTES>
__device__ __forceinline__ SplitTile split_tile(uint32_t tiles_m, uint32_t tiles_n, uint32_t splits, TensorArg<2>& x, TensorArg<2>& y, int32_t& k) {
  const uint32_t tiles = tiles_m * tiles_n, pos = xcd_contiguous(blockIdx.x, tiles * splits);
  SplitTile t;
  t.split = pos / tiles, t.tile = pos % tiles;
  grouped_tile(t.tile, tiles_m, tiles_n, &t.pm, &t.pn);
  const int32_t k_tiles = (min(min(x.shape[1], y.shape[0]), k) + BK - 1) / BK;
  const int32_t k0 = (int32_t)((int64_t)k_tiles * t.split / splits) * BK, k1 = (int32_t)((int64_t)k_tiles * (t.split + 1) / splits) * BK;
  x.ptr = (unsigned char*)x.ptr + (int64_t)k0 * BYTES;
  y.ptr = (unsigned char*)y.ptr + (int64_t)k0 * y.strides[0] * BYTES;
  x.shape[1] = max(0, min(x.shape[1], min(k, k1)) - k0);
  y.shape[0] = max(0, min(y.shape[0], min(k, k1)) - k0);
  k = min(x.shape[1], y.shape[0]);
  return t;
}

}  // namespace gemm
}  // namespace cutile
