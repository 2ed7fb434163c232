// Block-scaled products (MXFP8 and NVFP4, see mxfp8_gemm.hip and nvfp4_gemm.hip for the definitions) of few to medium many
// rows:  z[M,N] = alpha * sum_k x[i,k] sx[i,k/B] * y[j,k] sy[j,k/B].
//
// A wavefront reads 128-byte steps of its own 16-row blocks of x and y, eight lanes to a row so that every load instruction
// takes whole cache lines, keeps one to four steps in flight in registers, and turns each into matrix operands through a
// stage of LDS that no other wavefront touches: the K loop has no barrier.  Wavefronts divide the steps of K among
// themselves (and, for small outputs, among workgroups) and add up once at the end.
// Few rows are bound by the read of y and by the fixed cost of a launch whose every load leaves at once (mxfp8 1 x 14336 x 4096
// 39 -> 15 us, 16 x 4096 x 4096 29 -> 9.4; nvfp4 58 -> 11.5 and 53 -> 9.9), 64 and more by the L2 -> vector cache path, as each
// wavefront reads its x blocks for itself (nvfp4 200 x 14336 x 4096 70 -> 40 us).
// (Operands loaded in fragment order, one row to a lane, need no LDS but take the vector cache a clock per lane: 47 bytes/ns
// per compute unit, 128 x 4096 x 4096 mxfp8 89 us on 128 x 128 tiles.)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_common.h"
#include "kernel_args.h"
#include "split_k.h"

using namespace cutile;
using namespace cutile::gemm;

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// orders a wavefront's own LDS writes before its other lanes' reads (and reads before the next writes)
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// 8 wavefronts: WM x WN of them side by side on sub-tiles of 16 MB x 16 NB outputs, times WK on their own steps of K.  AHEAD
// steps are in flight per wavefront.  A step is 128 bytes of a row: 128 e4m3 values with four e8m0 scales, or (FP4) 256 e2m1
// values with sixteen e4m3 scales.
template <bool FP4, typename OutT, int MB, int NB, int WM, int WN, int WK, int AHEAD>
struct ScaledFlat {
  static constexpr int BM = 16 * MB * WM, BN = 16 * NB * WN, kThreads = WM * WN * WK * 64, PITCH = BN + 4;
  static constexpr int kRows = 16 * (MB + NB), kDataBytes = kRows * 128;   // of a wavefront's stage: y rows, then x rows
  static constexpr int kScaleRow = FP4 ? 16 : 4;                           // scale bytes of a step and row
  static constexpr int kStageBytes = kDataBytes + kRows * kScaleRow + 32;  // (reads for units past the end of K run over)
  static constexpr int kLoads = kRows / 8, kLdsBytes = 8 * kStageBytes > WK * BM * PITCH * 4 ? 8 * kStageBytes : WK * BM * PITCH * 4;
  static_assert(kThreads == 512 && NB == 4 && MB <= 4 && kLdsBytes <= 160 * 1024 - 64, "eight wavefronts, one load of 64 scale rows for y and one for x");

  __device__ static __forceinline__ int lds_off(int r, int u) { return r * 128 + ((u ^ ((r >> 1) & 7)) << 4); }

  __device__ static void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, const TensorArg<2>& xs, const TensorArg<2>& ys,
                             float alpha, float* partials, uint32_t* counters, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kLdsBytes];
    __shared__ uint32_t last;
    auto& red = *reinterpret_cast<float(*)[WK][BM][PITCH]>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN, l16 = lane & 15, grp = lane >> 4;
    // split-major order, bands of kGroupM tile rows inside: an XCD's contiguous share is neighbouring tiles on one range of K
    const uint32_t tiles = tiles_m * tiles_n, pos = xcd_contiguous(blockIdx.x, tiles * splits), split = pos / tiles, tile = pos % tiles;
    const uint32_t per_group = kGroupM * tiles_n, first_m = tile / per_group * kGroupM, group_rows = min(tiles_m - first_m, (uint32_t)kGroupM);
    const uint32_t pm = first_m + tile % per_group % group_rows, pn = tile % per_group / group_rows;
    const int32_t M = x.shape[0], N = y.shape[0], row_bytes = min(x.shape[1], y.shape[1]);
    const int32_t row0 = pm * BM, col0 = pn * BN;

    // Operands end below 2 GiB, so an offset with the top bit set reads 0: rows outside, and units past the end of a row.
    constexpr uint32_t kOob = 0x80000000u;
    auto rsrc = [](const TensorArg<2>& t) { return make_rsrc(t.ptr, (uint32_t)((int64_t)(t.shape[0] - 1) * t.strides[0] + t.shape[1])); };
    const __amdgpu_buffer_rsrc_t rx = rsrc(x), ry = rsrc(y), rsx = rsrc(xs), rsy = rsrc(ys);
    const int32_t wave_row = row0 + wm * MB * 16, wave_col = col0 + wn * NB * 16;
    uint32_t off[kLoads], s_off[2];   // load i: 8 rows, lane = (row, unit); scales: a row to a lane
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const bool is_y = i < NB * 2;
      const int32_t r = (is_y ? wave_col + i * 8 : wave_row + (i - NB * 2) * 8) + (lane >> 3);
      off[i] = r < (is_y ? N : M) ? (uint32_t)r * (uint32_t)(is_y ? y.strides[0] : x.strides[0]) + (lane & 7) * 16 : kOob;
    }
    s_off[0] = wave_col + lane < N ? (uint32_t)(wave_col + lane) * (uint32_t)ys.strides[0] : kOob;
    s_off[1] = lane < MB * 16 && wave_row + lane < M ? (uint32_t)(wave_row + lane) * (uint32_t)xs.strides[0] : kOob;
    const int32_t last_scales = row_bytes / 128 * kScaleRow + (FP4 ? row_bytes % 128 / 8 : 0) - kScaleRow;   // the last whole step's worth of a scale row

    struct InFlight {
      u32x4 data[kLoads];
      u32x4 sy, sx;   // (FP4: all four dwords)
    };
    auto fetch = [&](InFlight& f, int32_t step) {
      const int32_t at = step * 128;
      const uint32_t dead = at + (lane & 7) * 16 < row_bytes ? 0u : kOob;
#pragma unroll
      for (int i = 0; i < kLoads; ++i) f.data[i] = __builtin_amdgcn_raw_buffer_load_b128(i < NB * 2 ? ry : rx, (off[i] + at) | dead, 0, 0);
      const int32_t s_at = min(step * kScaleRow, last_scales);
      if constexpr (FP4) {
        f.sy = __builtin_amdgcn_raw_buffer_load_b128(rsy, s_off[0] + s_at, 0, 0);
        f.sx = __builtin_amdgcn_raw_buffer_load_b128(rsx, s_off[1] + s_at, 0, 0);
      } else {
        f.sy.x = __builtin_amdgcn_raw_buffer_load_b32(rsy, s_off[0] + s_at, 0, 0);
        f.sx.x = __builtin_amdgcn_raw_buffer_load_b32(rsx, s_off[1] + s_at, 0, 0);
      }
    };
    unsigned char* const stage = lds + wave * kStageBytes;
    unsigned char* const s_stage = stage + kDataBytes;
    auto put = [&](const InFlight& f) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) *reinterpret_cast<u32x4*>(stage + lds_off(i * 8 + (lane >> 3), lane & 7)) = f.data[i];
      if constexpr (FP4) {
        *reinterpret_cast<u32x4*>(s_stage + lane * 16) = f.sy;
        if (lane < MB * 16) *reinterpret_cast<u32x4*>(s_stage + (64 + lane) * 16) = f.sx;
      } else {
        *reinterpret_cast<uint32_t*>(s_stage + lane * 4) = f.sy.x;
        if (lane < MB * 16) *reinterpret_cast<uint32_t*>(s_stage + (64 + lane) * 4) = f.sx.x;
      }
    };

    f32x4 acc[NB][MB];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[n][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Blocks 0 .. NB - 1 of the stage are y, then x; a lane reads units grp and 4 + grp of its row.
    auto unit = [&](int block, int h) { return *reinterpret_cast<const u32x4*>(stage + lds_off(l16, 4 * h + grp) + block * (16 * 128)); };
    auto multiply_fp8 = [&] {
      auto frag = [&](int block) {
        const u32x4 a = unit(block, 0), b = unit(block, 1);
        return i32x8{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, (int)b.z, (int)b.w};
      };
      auto scale = [&](int block) { return (int)s_stage[(block * 16 + l16) * 4 + grp]; };   // lanes of group g supply the scale of block g
      i32x8 fx[MB];
      int sx[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m) sx[m] = scale(NB + m), fx[m] = frag(NB + m);
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const int sy = scale(n);
        const i32x8 fy = frag(n);
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[n][m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fy, fx[m], acc[n][m], 0, 0, 0, sy, 0, sx[m]);
      }
    };
    // Expanded to f16 (exact: at most six significant bits); dword d of a unit is one K group of 8 of v_mfma_f32_16x16x32_f16,
    // the same positions of x and y in the same lane, so the order of K does not matter.
    auto expand = [](uint32_t packed, f16x2 s) {
      const f16x2 v[4] = {__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 0) * s, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 1) * s,
                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 2) * s, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 3) * s};
      return f16x8{v[0][0], v[0][1], v[1][0], v[1][1], v[2][0], v[2][1], v[3][0], v[3][1]};
    };
    auto multiply_fp4 = [&](int32_t step) {
      const int32_t shift = step * kScaleRow - min(step * kScaleRow, last_scales);   // where the step begins in the scales that were read
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int32_t u = 4 * h + grp;
        const bool live = step * 128 + u * 16 < row_bytes;
        const int at = live ? 2 * u + shift : 0;
        auto scales = [&](int block) -> uint32_t {   // two scale bytes of the unit; 0 past the end of K (a foreign scale may be NaN)
          const uint32_t v = *reinterpret_cast<const uint16_t*>(s_stage + (block * 16 + l16) * 16 + at);
          return live ? v : 0u;
        };
        auto pair = [](uint32_t two, auto byte) {
          const _Float16 s = (_Float16)__builtin_amdgcn_cvt_f32_fp8((int)two, decltype(byte)::value);   // e4m3 -> f32 -> f16: exact
          return f16x2{s, s};
        };
        u32x4 ux[MB];
        uint32_t sx[MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) sx[m] = scales(NB + m), ux[m] = unit(NB + m, h);
        u32x4 uy[NB];
        uint32_t sy[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) sy[n] = scales(n), uy[n] = unit(n, h);
        auto half = [&](auto byte) {   // dwords 2 byte and 2 byte + 1: one scale
          constexpr int B = decltype(byte)::value;
#pragma unroll
          for (int d = 2 * B; d < 2 * B + 2; ++d) {
            f16x8 fx[MB];
#pragma unroll
            for (int m = 0; m < MB; ++m) fx[m] = expand(ux[m][d], pair(sx[m], byte));
#pragma unroll
            for (int n = 0; n < NB; ++n) {
              const f16x8 fy = expand(uy[n][d], pair(sy[n], byte));
#pragma unroll
              for (int m = 0; m < MB; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fy, fx[m], acc[n][m], 0, 0, 0);
            }
          }
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
        __builtin_amdgcn_sched_barrier(0);   // the operands of one unit at a time, or registers spill
      }
    };

    // step s belongs to share s % stride of the wavefronts; steps past the end fetch zeros, which add nothing
    const int32_t steps = (row_bytes + 127) / 128, stride = WK * (int32_t)splits;
    const int32_t first = (int32_t)split * WK + wk;
    InFlight f[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(f[i], first + i * stride);
    for (int32_t s = first; s < steps; s += AHEAD * stride) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const int32_t step = s + i * stride;
        wave_fence();
        __builtin_amdgcn_sched_barrier(0);
        put(f[i]);
        wave_fence();
        __builtin_amdgcn_sched_barrier(0);
        fetch(f[i], step + AHEAD * stride);
        __builtin_amdgcn_sched_barrier(0);   // the loads leave before the products
        if constexpr (FP4)
          multiply_fp4(step);
        else
          multiply_fp8();
      }
    }
    __syncthreads();   // the stages become the partial sums

    // lane (grp, l16) holds row l16 of block m and columns 4 grp .. + 3 of block n
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < NB; ++n) *reinterpret_cast<f32x4*>(&red[wk][(wm * MB + m) * 16 + l16][(wn * NB + n) * 16 + grp * 4]) = acc[n][m];
    __syncthreads();
    constexpr int kQuads = BN / 4;
    const int32_t rows = min(BM, z.shape[0] - row0), zn = z.shape[1];
    OutT* const zp = (OutT*)z.ptr;
    auto sum = [&](int o4) {
      f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][o4 / kQuads][o4 % kQuads * 4]);
#pragma unroll
      for (int w = 1; w < WK; ++w) v += *reinterpret_cast<const f32x4*>(&red[w][o4 / kQuads][o4 % kQuads * 4]);
      return v;
    };
    auto store = [&](int o4, f32x4 v) {   // z rows are 16-byte aligned quads of columns
      const int32_t c = col0 + o4 % kQuads * 4;
      if (c >= zn) return;
      OutT* dst = zp + (int64_t)(row0 + o4 / kQuads) * z.strides[0] + c;
      if constexpr (sizeof(OutT) == 2)
        *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16x2(v[0] * alpha, v[1] * alpha), pack_bf16x2(v[2] * alpha, v[3] * alpha)};
      else
        *reinterpret_cast<f32x4*>(dst) = f32x4{v[0] * alpha, v[1] * alpha, v[2] * alpha, v[3] * alpha};
    };
    if (splits == 1) {
      for (int o4 = tid; o4 < rows * kQuads; o4 += kThreads) store(o4, sum(o4));
      return;
    }
    const BlockPartials part(partials + (int64_t)tile * splits * (BM * BN), BM * BN * 4, splits);
    for (int o4 = tid; o4 < rows * kQuads; o4 += kThreads) part.store(split, o4, sum(o4));
    if (!last_to_arrive(counters + tile, splits, &last)) return;
    part.add_up<kThreads, (BM * kQuads > kThreads ? 2 : 1)>(rows * kQuads, store);
  }
};

}  // namespace

#define SCALED_FLAT_KERNEL(ENTRY, NAME, FP4, OUT_T, MB, NB, WM, WN, WK, AHEAD)                                                        \
  extern "C" __global__ void __launch_bounds__(512)                                                                                   \
      ENTRY##__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, TensorArg<2> xs, TensorArg<2> ys, float alpha, float* partials, \
                      uint32_t* counters, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits) {                                      \
    ScaledFlat<FP4, OUT_T, MB, NB, WM, WN, WK, AHEAD>::run(z, x, y, xs, ys, alpha, partials, counters, tiles_m, tiles_n, splits);      \
  }
#define SCALED_FLAT_FAMILY(ENTRY, PREFIX, FP4, OUT_T, AHEAD16, AHEAD32, AHEAD64)       \
  SCALED_FLAT_KERNEL(ENTRY, PREFIX##_flat16x64, FP4, OUT_T, 1, 4, 1, 1, 8, AHEAD16)    \
  SCALED_FLAT_KERNEL(ENTRY, PREFIX##_flat32x64, FP4, OUT_T, 2, 4, 1, 1, 8, AHEAD32)    \
  SCALED_FLAT_KERNEL(ENTRY, PREFIX##_flat64x64, FP4, OUT_T, 4, 4, 1, 1, 8, AHEAD64)    \
  SCALED_FLAT_KERNEL(ENTRY, PREFIX##_flat64x128, FP4, OUT_T, 4, 4, 1, 2, 4, AHEAD64)   \
  SCALED_FLAT_KERNEL(ENTRY, PREFIX##_flat128x128, FP4, OUT_T, 4, 4, 2, 2, 2, AHEAD64)
SCALED_FLAT_FAMILY(linear_tile_entry, mxfp8_bf16, false, __bf16, 2, 2, 1)
SCALED_FLAT_FAMILY(linear_tile_entry, mxfp8_f32, false, float, 2, 2, 1)
SCALED_FLAT_FAMILY(linear_tile_nvfp4_entry, bf16, true, __bf16, 2, 2, 1)
SCALED_FLAT_FAMILY(linear_tile_nvfp4_entry, f32, true, float, 2, 2, 1)
