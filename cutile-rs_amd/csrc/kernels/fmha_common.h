// What the attention kernels share: 16-bit element types, the exchange between the lanes of a query row, the order of the workgroups.
#pragma once
#include <hip/hip_runtime.h>

#include "kernel_args.h"
#include "lane_exchange.h"

using namespace cutile;

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define LDS_PTR(T) __attribute__((address_space(3))) T*

constexpr float kLog2e = 1.4426950408889634f;

// Bytes from the first element of row 0 to the last of row rows - 1 (16-bit elements, `row_stride`
// elements apart, `d` per row); nothing for an empty range, so that every access is out of range.
__device__ __forceinline__ uint32_t rows_extent_bytes(int32_t rows, int32_t row_stride, int32_t d) {
  return rows > 0 ? (uint32_t)(((int64_t)(rows - 1) * row_stride + d) * 2) : 0u;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

template <typename T>
struct Elem;
template <>
struct Elem<__bf16> {
  using vec8 = bf16x8;
  __device__ static __forceinline__ f32x16 mfma(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, b2));  // v_cvt_pk_bf16_f32, RNE
  }
};
template <>
struct Elem<_Float16> {
  using vec8 = f16x8;
  __device__ static __forceinline__ f32x16 mfma(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, h2));  // v_cvt_pk_f16_f32
  }
};

// The two lanes that own one query row are 32 apart: their maximum and sum go through v_permlane32_swap, and the
// four lanes of a head in the matrix-core decode kernel through v_permlane16_swap first (lane_exchange.h), inside the
// vector ALU, where a lane-indexed permute would cost a trip through the LDS crossbar and a wait of its own in the middle
// of every softmax segment.
__device__ __forceinline__ float max_across_halves(float v) { return lanes::across_halves<lanes::Max>(v); }
__device__ __forceinline__ float sum_across_halves(float v) { return lanes::across_halves<lanes::Sum>(v); }
__device__ __forceinline__ float max_across_rows(float v) { return lanes::across_rows<lanes::Max>(v); }
__device__ __forceinline__ float sum_across_rows(float v) { return lanes::across_rows<lanes::Sum>(v); }

// (batch*head, query tile) of this workgroup.  Workgroups are dealt round-robin to
// the 8 XCDs in dispatch order; every query tile of one head is given to the same
// XCD, consecutively, so that the head's K and V (read by each of its query
// tiles) stay in that XCD's L2 instead of being fetched from HBM once per tile.
// Causal launches do the same with a few heads side by side per XCD, heaviest tiles
// first (see below); one head at a time measured slower than the plain order because the
// last head's long tiles start late.
__device__ __forceinline__ void head_and_tile(uint32_t n_bh, uint32_t n_qt, int32_t causal, uint32_t group, int32_t* bh, int32_t* q_tile) {
  constexpr uint32_t kNumXcd = 8;
  const uint32_t id = blockIdx.x + gridDim.x * blockIdx.y;
  uint32_t b, t;
  constexpr uint32_t kCusPerXcd = 32;
  uint32_t side = n_qt >= kCusPerXcd ? 1 : kCusPerXcd / n_qt;     // heads an XCD works on side by side
  // Query heads that share a KV head (consecutive, `group` of them) run side by side on one XCD, tile for tile, so
  // that the K/V rows one of them fetches serve all of them.
  if (group > 1) side = (side + group - 1) / group * group;
  if (n_bh % kNumXcd == 0 && !causal && group <= 1) {
    const uint32_t xcd = id % kNumXcd, slot = id / kNumXcd;
    b = (slot / n_qt) * kNumXcd + xcd;
    t = slot % n_qt;
  } else if (n_bh % (kNumXcd * side) == 0 && (causal || group > 1)) {
    // Causal tiles differ n_qt-fold in length.  An XCD takes `side` heads at a time (their K/V fit its L2) and
    // walks their tiles heaviest first, heads interleaved: the compute units that drew the short tiles of one
    // group free up first and draw the long tiles of the next, so lengths pair up (n_qt + 1 per two tiles).
    const uint32_t xcd = id % kNumXcd, slot = id / kNumXcd, per_group = side * n_qt;
    b = xcd * (n_bh / kNumXcd) + (slot / per_group) * side + (slot % per_group) % side;
    t = (slot % per_group) / side;
  } else {   // plain order: every (head, tile) still covered exactly once
    b = id % n_bh;
    t = id / n_bh;
  }
  *bh = (int32_t)b;
  *q_tile = causal ? (int32_t)(n_qt - 1 - t) : (int32_t)t;
}

}  // namespace
