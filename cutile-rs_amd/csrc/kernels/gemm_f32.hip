// f32 GEMM on the matrix cores: z[M,N] (+)= x[M,K] . y[K,N], every product and sum in f32 (v_mfma_f32_16x16x4_f32).
//
// The matrix instruction does 64 f32 flops a clock and SIMD, a sixteenth of the 16-bit rate, so operands are cheap against it and
// need no LDS: a wavefront of 64 x 64 outputs reads 8 KiB for 2048 clocks of matrix work, which the vector cache and L2 deliver beside it.
// A workgroup owns a strip of 64 columns by 16, 32 or 64 rows; its 8 wavefronts and gridDim.z workgroups of the same strip share K, step
// by step, and their partial sums meet once, after the last step.  A lane reads 4 consecutive columns of 4 K rows of y (16 lanes cover
// 64 columns, the four lane groups 16 K rows) and 4 consecutive K values of a row of x.  Column j of all 16 lanes is a column set of
// its own, so each register of a y read is an operand as it stands, and any assignment of K positions to lanes will do if x and y agree:
// register i of lane group g is K position 4 g + i.  The MFMA is issued with y first, so a lane ends up with 16 consecutive columns of a row.
//
// With few rows the product is a read of y (3 x 2160 x 2208: 9.9 us), with many the matrix pipes bound it (677 x 1941 x 4357: 169 us, 68
// TFLOP/s): a strip's sums through LDS and its last round of workgroups are the rest.  Tiles of 128 x 128 and 128 x 256 with K on two and one
// wavefronts were no faster at any K beyond 128 (1541 x 2160 x 512: 53.4 us here, 55.8 on 128 x 128).
// Errors against 64 bits are 0.29 to 0.86 of the any-layout kernel's (K from 8192 to 32), which adds K up in one chain.
#include <hip/hip_runtime.h>

#include "gemm_common.h"
#include "kernel_args.h"
#include "split_k.h"

using namespace cutile;
using namespace cutile::gemm;

namespace {

template <int MB>
struct GemmF32 {
  static constexpr int ROWS = 16 * MB, COLS = 64, WAVES = 8;
  static constexpr int PITCH = COLS + 4;                         // floats of one row of partial sums: 16 rows written by one instruction spread over the banks
  static constexpr int H = MB <= 2 ? 2 : 1, KS = 16 * H;         // K positions of a step: two of them are in flight, in registers

  struct Step {
    f32x4 y[H][4], x[H][MB];
  };
  __device__ static __forceinline__ f32x4 load(const float* p) {   // any 4-byte boundary
    f32x4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 4), 16);
    return v;
  }

  __device__ static void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, int32_t k_total, int32_t cover_m,
                             int32_t cover_n, int32_t accumulate, float* partials, uint32_t* counters, uint32_t tiles_m, uint32_t tiles_n) {
    __shared__ __attribute__((aligned(16))) float red[WAVES][ROWS][PITCH];
    __shared__ uint32_t last;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, grp = lane >> 4;
    const int32_t M = x.shape[0], N = y.shape[1];
    const int64_t lda = x.strides[0], ldb = y.strides[0];
    const int32_t k_valid = min(min(x.shape[1], y.shape[0]), k_total);
    const uint32_t tile = xcd_contiguous(blockIdx.x, tiles_m * tiles_n);   // (strips on the x axis alone: y holds 65535 of them)
    uint32_t pm, pn;
    grouped_tile(tile, tiles_m, tiles_n, &pm, &pn);
    const int32_t row0 = (int32_t)pm * ROWS;
    const int32_t col_first = (int32_t)pn * COLS;                                // first column this workgroup stores
    const int32_t col0 = min(col_first, N - COLS);                               // the last strip is moved back to lie inside y (N >= 64)

    const float* yp = (const float*)y.ptr + col0 + l16 * 4 + (int64_t)(grp * 4) * ldb;
    const float* xp[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)   // rows past the end repeat the last one; their results are not stored
      xp[mb] = (const float*)x.ptr + (int64_t)min(row0 + mb * 16 + l16, M - 1) * lda + grp * 4;

    f32x4 acc[4][MB];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto fetch = [&](Step& s, int32_t step) {
      const int64_t k0 = (int64_t)step * KS;
#pragma unroll
      for (int h = 0; h < H; ++h) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s.y[h][i] = load(yp + (k0 + h * 16 + i) * ldb);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) s.x[h][mb] = load(xp[mb] + k0 + h * 16);
      }
    };
    auto multiply = [&](const Step& s) {
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) acc[j][mb] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.y[h][i][j], s.x[h][mb][i], acc[j][mb], 0, 0, 0);
    };

    // step s of the K loop belongs to wavefront s % stride of the strip
    const int32_t steps = k_valid / KS, stride = WAVES * gridDim.z;
    int32_t s = blockIdx.z * WAVES + wave;
    const int32_t own = s;
    Step a, b;
    if (s < steps) fetch(a, s);
    for (; s + stride < steps; s += 2 * stride) {
      fetch(b, s + stride);
      __builtin_amdgcn_sched_barrier(0);   // a whole step is in flight while the one before it is multiplied
      multiply(a);
      if (s + 2 * stride < steps) fetch(a, s + 2 * stride);
      __builtin_amdgcn_sched_barrier(0);
      multiply(b);
    }
    if (s < steps) multiply(a);
    if (k_valid % KS != 0 && steps % stride == own) {   // the ragged last step: K positions past the end are 0 on both sides
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int32_t k = steps * KS + h * 16 + grp * 4 + i, back = max(0, k - (k_valid - 1));   // read at the last position, then cleared
          const f32x4 v = load(yp + (int64_t)(k - grp * 4 - back) * ldb);
          a.y[h][i] = back ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : v;
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            const float e = xp[mb][k - grp * 4 - back];
            a.x[h][mb][i] = back ? 0.0f : e;
          }
        }
      multiply(a);
    }

    // lane (grp, l16) holds, for row block mb, row l16 and the columns 16 grp + 4 i + j of the strip in acc[j][mb][i]
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(&red[wave][mb * 16 + l16][16 * grp + 4 * i]) = f32x4{acc[0][mb][i], acc[1][mb][i], acc[2][mb][i], acc[3][mb][i]};
    __syncthreads();
    const int32_t quads = min(ROWS, cover_m - row0) * (COLS / 4);   // four consecutive columns of a row to a thread
    auto wave_sum = [&](int o) {
      const int r = o / (COLS / 4), c = o % (COLS / 4) * 4;
      f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][r][c]);
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v += *reinterpret_cast<const f32x4*>(&red[w][r][c]);
      return v;
    };
    float* const zp = (float*)z.ptr;
    auto store = [&](int o, f32x4 v) {
      const int32_t gc = col0 + o % (COLS / 4) * 4;
      float* dst = zp + (int64_t)(row0 + o / (COLS / 4)) * z.strides[0] + gc;
      if (gc >= col_first && gc + 4 <= cover_n) {
        if (accumulate) v += load(dst);
        __builtin_memcpy(__builtin_assume_aligned(dst, 4), &v, 16);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (gc + e >= col_first && gc + e < cover_n) {
            const float f = v[e];
            dst[e] = accumulate ? f + dst[e] : f;
          }
      }
    };
    const uint32_t splits = gridDim.z;
    if (splits == 1) {
      for (int o = tid; o < quads; o += WAVES * 64) store(o, wave_sum(o));
      return;
    }
    const BlockPartials part(partials + (int64_t)tile * splits * (ROWS * COLS), ROWS * COLS * 4, splits);
    for (int o = tid; o < quads; o += WAVES * 64) part.store(blockIdx.z, o, wave_sum(o));
    if (!last_to_arrive(counters + tile, splits, &last)) return;
    part.add_up<WAVES * 64, (ROWS * COLS / 4 > WAVES * 64 ? 2 : 1)>(quads, store);
  }
};

}  // namespace

#define GEMM_F32_KERNEL(NAME, MB)                                                                                                   \
  extern "C" __global__ void __launch_bounds__(512)                                                                                 \
      gemm_entry__f32_##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k_total, int32_t cover_m, int32_t cover_n,   \
                             int32_t accumulate, float* partials, uint32_t* counters, uint32_t tiles_m, uint32_t tiles_n) {         \
    GemmF32<MB>::run(z, x, y, k_total, cover_m, cover_n, accumulate, partials, counters, tiles_m, tiles_n);                          \
  }
GEMM_F32_KERNEL(strip16x64, 1)
GEMM_F32_KERNEL(strip32x64, 2)
GEMM_F32_KERNEL(strip64x64, 4)
