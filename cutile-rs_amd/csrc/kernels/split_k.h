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
constexpr int kAgentScope = 16;   // buffer accesses with sc1: past the L2, which the XCDs do not share
// 16 bytes of a partial sum.  No scalar offset: a 16-byte store that has one reads its data registers for some cycles after it issues, and the
// compiler, which guards only the other form, may reuse them in the next instruction.
__device__ __forceinline__ void store_partial(f32x4 v, __amdgpu_buffer_rsrc_t to, uint32_t at) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), to, at, 0, kAgentScope);
}
// The partial sums of one block: quads of four neighbouring outputs, numbered as the kernel likes, one copy of `bytes` per split.
struct BlockPartials {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t bytes, splits;

  __device__ __forceinline__ BlockPartials(float* mine, uint32_t block_bytes, uint32_t n) : rsrc(make_rsrc(mine, block_bytes * n)), bytes(block_bytes), splits(n) {}
  __device__ __forceinline__ void store(uint32_t split, int quad, f32x4 v) const {
    store_partial(v, rsrc, split * bytes + quad * 16);
  }
  // take(quad, sum in split order) for every quad, dealt to THREADS threads, Q quads of eight splits at a time: a read past the L2 takes about a
  // microsecond, and one after another (a value, a split) they were much of a launch of few rows (f16, kernel time in us with such reads and
  // here, K shared by 6 or 7: 17 x 1088 x 7168 13.5, 8.9; 37 x 2048 x 6656 21.5, 15.0; 64 x 2048 x 6656 on 64 x 64 tiles, by 8, 20.5, 16.4).
  template <int THREADS, int Q, typename F>
  __device__ __forceinline__ void add_up(int quads, F&& take) const {
    constexpr uint32_t kOob = 0x80000000u, kAtOnce = 8;
    for (int o = threadIdx.x; o < quads; o += THREADS * Q) {
      f32x4 sum[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) sum[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
      for (uint32_t k = 0; k < splits; k += kAtOnce) {
        u32x4 v[kAtOnce][Q];
#pragma unroll
        for (uint32_t i = 0; i < kAtOnce; ++i)
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            const bool wanted = k + i < splits && o + q * THREADS < quads;   // others read 0 and never leave the compute unit
            v[i][q] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, wanted ? (uint32_t)(o + q * THREADS) * 16 : kOob, k + i < splits ? (k + i) * bytes : 0, kAgentScope);
          }
#pragma unroll
        for (uint32_t i = 0; i < kAtOnce; ++i)
#pragma unroll
          for (int q = 0; q < Q; ++q) sum[q] += __builtin_bit_cast(f32x4, v[i][q]);
      }
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (o + q * THREADS < quads) take(o + q * THREADS, sum[q]);
    }
  }
};
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
template <int TM, int TN, int THREADS>
__device__ __forceinline__ bool combine_tile(f32x4 (&acc)[TN][TM], float* mine, uint32_t* counter, uint32_t split, uint32_t splits, uint32_t* shared_flag) {
  constexpr uint32_t kTile = TM * TN * THREADS * 16;   // bytes
  const __amdgpu_buffer_rsrc_t part = make_rsrc(mine, kTile * splits);
#pragma unroll
  for (int r = 0; r < TM * TN; ++r)
    store_partial(acc[r % TN][r / TN], part, split * kTile + r * (THREADS * 16) + threadIdx.x * 16);
  if (!last_to_arrive(counter, splits, shared_flag)) return false;
  // (one partial tile at a time: with the next one's loads in flight beside it 48 and 54 tiles of 128 x 128 took 14.5 us where they take 13.7)
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
