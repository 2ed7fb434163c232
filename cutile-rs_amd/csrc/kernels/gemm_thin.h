// GEMM of few rows: strips of columns, y streamed through registers (gemm_small.hip, gemm_tiles.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_common.h"
#include "kernel_args.h"
#include "split_k.h"

namespace cutile {
namespace gemm {

// ---- few rows: y streams through registers once -------------------------------------------------------------------------
// With at most 64 rows of x the product is a read of y (2 K N bytes), and a 128-row tile per workgroup reads it at a
// fraction of the HBM rate: N / 128 workgroups, each waiting for one K tile after another (M = 1, K = N = 4096, f16:
// 51 us, 0.66 TB/s).  Here a workgroup owns a strip of CW = 16 CPL columns, and K is dealt in steps of 64 rows to its
// wavefronts and to gridDim.z workgroups of the same strip; the partial sums meet once, after the last step.  No barrier
// and no LDS inside the loop: a lane reads CPL consecutive columns of 8 consecutive K rows (16 lanes cover a row of the
// strip, the four lane groups 32 rows), and since column j of all 16 lanes is a column set of its own, v_perm turns the
// 8 x CPL values into CPL operands of v_mfma_f32_16x16x32 (any assignment of columns to MFMA rows will do, the
// store undoes it).  What bounds a compute unit is the number of cache lines it can have in flight (its 32 KiB vector
// cache: 256 lines), so a strip is never narrower than a 128-byte line: 32-column strips read 17-22 bytes/ns per compute
// unit, 64-column ones 26-38, 128-column ones up to 53; and x is read two 32-wide steps at a time for the same reason.
// NT: y past the caches, for a y that is read once and too large to be found there again (96 MiB and more, 16 rows at most): a streaming
// read of plain loads fills them first.  f16, one row, weights from memory, us: 4096 x 14336 24.3 -> 22.0 on 128-column strips (64-column ones
// 23.0), 14336 x 4096 24.7 -> 23.4, 8192 x 28672 83.0 -> 75.0; a block of one new token over these weights 131 -> 120.  The price: weights that
// the memory-side cache (256 MB) still holds when they are read again are read slower (one row, plain and NT: 14336 x 4096 again at once 20.4, 22.0,
// two of them in turn 20.5, 22.7, four 24.9, 23.2; 8192 x 12288, 201 MB, 31.5, 34.3, two 38.9, 35.6; 8192 x 16384, 268 MB, 41.8, 45.9, two 50.4,
// 47.1; 8192 x 20480, 336 MB, 63.1, 58.9).  A program that steps through layers of such weights has read more than that cache holds
// before it comes back to one.  Not for 17 to 32 rows, where it gains 2 to 3 % and costs 16 to 32 %, nor for smaller weights, several of which fit.
template <typename InT, typename OutT, int MB, int CPL, int WAVES, bool NT>
struct GemmThin {
  static constexpr int CW = 16 * CPL, ROWS = 16 * MB, kThreads = WAVES * 64;
  static constexpr int PITCH = CW + 4;      // floats of one row of partial sums: 16 rows written by one instruction spread over the banks
  static constexpr int CU32 = CPL / 2;      // registers of one K row

  struct Step {                             // 64 K rows
    uint32_t y[2][8][CU32];
    u32x4 x[2][MB];
  };

  // Rows start on any 2-byte boundary (an odd N or K): global memory takes every alignment at the width of the access.
  template <int BYTES>
  __device__ static __forceinline__ void load(const unsigned char* p, uint32_t* into) {
    __builtin_memcpy(into, __builtin_assume_aligned(p, 2), BYTES);
  }

  __device__ static __forceinline__ void load_y(const unsigned char* p, uint32_t* into) {
    if constexpr (NT) {
      typedef uint32_t vec __attribute__((ext_vector_type(CU32), aligned(2)));
      const vec v = __builtin_nontemporal_load(reinterpret_cast<const vec*>(p));
#pragma unroll
      for (int c = 0; c < CU32; ++c) into[c] = v[c];
    } else {
      load<CPL * 2>(p, into);
    }
  }

  __device__ static void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, int32_t k_total, int32_t cover_m,
                             int32_t cover_n, int32_t accumulate, float* partials, uint32_t* counters) {
    __shared__ __attribute__((aligned(16))) float red[WAVES][ROWS][PITCH];
    __shared__ uint32_t last;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, grp = lane >> 4;
    const int32_t M = x.shape[0], N = y.shape[1];
    const int64_t lda = (int64_t)x.strides[0] * 2, ldb = (int64_t)y.strides[0] * 2;   // bytes
    const int32_t k_valid = min(min(x.shape[1], y.shape[0]), k_total);
    const int32_t strip = xcd_contiguous(blockIdx.x, gridDim.x);
    const int32_t col_first = strip * CW;              // first column this workgroup stores
    const int32_t col0 = min(col_first, N - CW);       // the last strip is moved back to lie inside y (N >= CW)
    const int32_t row0 = blockIdx.y * ROWS;

    const unsigned char* yp = (const unsigned char*)y.ptr + (int64_t)col0 * 2;
    const uint32_t y_lane = (uint32_t)(l16 * CPL * 2) + (uint32_t)(grp * 8) * (uint32_t)ldb;   // < 32 ldb: operands end below 2 GiB
    const unsigned char* xp[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)   // rows past the end repeat the last one; their results are not stored
      xp[mb] = (const unsigned char*)x.ptr + (int64_t)min(row0 + mb * 16 + l16, M - 1) * lda + grp * 16;

    f32x4 acc[CPL][MB];
#pragma unroll
    for (int j = 0; j < CPL; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto fetch = [&](Step& s, int32_t step) {
      const unsigned char* base = yp + (int64_t)step * (64 * ldb);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) load_y(base + (h * 32 + i) * ldb + y_lane, s.y[h][i]);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) load<16>(xp[mb] + (int64_t)step * 128 + h * 64, reinterpret_cast<uint32_t*>(&s.x[h][mb]));
      }
    };
    auto multiply = [&](const Step& s) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
          u32x4 f;
#pragma unroll
          for (int p = 0; p < 4; ++p)
            f[p] = __builtin_amdgcn_perm(s.y[h][2 * p + 1][j / 2], s.y[h][2 * p][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[j][mb] = mfma_16x16x32<InT>(__builtin_bit_cast(bf16x8, f), __builtin_bit_cast(bf16x8, s.x[h][mb]), acc[j][mb]);
        }
    };

    // step s of the K loop belongs to wavefront s % stride of the strip
    const int32_t steps = k_valid / 64, stride = WAVES * gridDim.z;
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
    if (k_valid % 64 != 0 && steps % stride == own) {   // the ragged last step: K positions past the end are 0 on both sides
      const int32_t k0 = steps * 64;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int32_t k = k0 + h * 32 + grp * 8 + i;
          load<CPL * 2>(yp + (int64_t)min(k, k_valid - 1) * ldb + l16 * CPL * 2, a.y[h][i]);
#pragma unroll
          for (int c = 0; c < CU32; ++c) a.y[h][i][c] = k < k_valid ? a.y[h][i][c] : 0u;
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const uint16_t* row = reinterpret_cast<const uint16_t*>(xp[mb] - grp * 16);
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            uint32_t e[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const int32_t k = k0 + h * 32 + grp * 8 + 2 * p + i;
              e[i] = row[min(k, k_valid - 1)];
              e[i] = k < k_valid ? e[i] : 0u;
            }
            a.x[h][mb][p] = e[0] | (e[1] << 16);
          }
        }
      }
      multiply(a);
    }

    // lane (grp, l16) holds, for row block mb, row l16 and the columns CPL * (4 grp + i) + j of the strip
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      if (row0 + mb * 16 + l16 < cover_m) {
        float* row = &red[wave][mb * 16 + l16][CPL * 4 * grp];
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[(4 * q + e) % CPL][mb][(4 * q + e) / CPL];
          *reinterpret_cast<f32x4*>(row + 4 * q) = v;
        }
      }
    __syncthreads();
    const int32_t quads = min(ROWS, cover_m - row0) * (CW / 4);   // four consecutive columns of a row to a thread
    auto wave_sum = [&](int o) {
      const int r = o / (CW / 4), c = o % (CW / 4) * 4;
      f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += *reinterpret_cast<const f32x4*>(&red[w][r][c]);
      return v;
    };
    OutT* zp = (OutT*)z.ptr;
    auto store = [&](int o, f32x4 v) {
      const int32_t gc = col0 + o % (CW / 4) * 4;
      OutT* dst = zp + (int64_t)(row0 + o / (CW / 4)) * z.strides[0] + gc;
      if (gc >= col_first && gc + 4 <= cover_n) {
        OutT e[4];
        if (accumulate) __builtin_memcpy(e, __builtin_assume_aligned(dst, sizeof(OutT)), sizeof(e));
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = (OutT)(accumulate ? v[i] + (float)e[i] : v[i]);
        __builtin_memcpy(__builtin_assume_aligned(dst, sizeof(OutT)), e, sizeof(e));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (gc + i >= col_first && gc + i < cover_n) dst[i] = (OutT)(accumulate ? v[i] + (float)dst[i] : v[i]);
      }
    };
    const uint32_t splits = gridDim.z;
    if (splits == 1) {
      if constexpr (ROWS == 16) {   // a value to a thread: quads of a row or two are 16 to 32 threads' work (1 x 299 x 1363 6.33 us, in quads 6.54: up to two rows and K = 1500 2 to 4 % of a launch)
        for (int o = tid; o < quads * 4; o += kThreads) {
          const int r = o / CW, c = o % CW, gc = col0 + c;
          if (gc < col_first || gc >= cover_n) continue;
          float v = 0.0f;
#pragma unroll
          for (int w = 0; w < WAVES; ++w) v += red[w][r][c];
          OutT* dst = zp + (int64_t)(row0 + r) * z.strides[0] + gc;
          if (accumulate) v += (float)*dst;
          *dst = (OutT)v;
        }
      } else {
        for (int o = tid; o < quads; o += kThreads) store(o, wave_sum(o));
      }
      return;
    }
    const uint32_t block = blockIdx.y * gridDim.x + strip;
    const BlockPartials part(partials + (int64_t)block * splits * (ROWS * CW), ROWS * CW * 4, splits);
    for (int o = tid; o < quads; o += kThreads) part.store(blockIdx.z, o, wave_sum(o));
    if (!last_to_arrive(counters + block, splits, &last)) return;
    part.add_up<kThreads, (ROWS * CW / 4 > kThreads ? 2 : 1)>(quads, store);
  }
};

}  // namespace gemm
}  // namespace cutile

#define GEMM_THIN_KERNEL(NAME, IN_T, OUT_T, MB, CPL, NT)                                                                            \
  extern "C" __global__ void __launch_bounds__(512)                                                                                 \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k_total, int32_t cover_m, int32_t cover_n,       \
                         int32_t accumulate, float* partials, uint32_t* counters) {                                                 \
    GemmThin<IN_T, OUT_T, MB, CPL, 8, NT>::run(z, x, y, k_total, cover_m, cover_n, accumulate, partials, counters);                  \
  }
