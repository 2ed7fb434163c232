// GEMM tiles whose rows may start on any 2-byte boundary: the output of such a tile, and the 256 x 256 form.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_common.h"
#include "kernel_args.h"

namespace cutile {
namespace gemm {

// ---- a K tile of 64 of register-staged tiles in LDS ------------------------------------------------------------------------------
// Byte offsets of 16-byte unit u of row r of the x tile (eight units a row) and of the y tile (UB), and a load from any 2-byte boundary.
template <int BN>
struct StagedLayout {
  static constexpr int BK = 64, UB = BN / 8;
  __device__ static __forceinline__ int a_lds_off(int r, int u) { return r * (BK * 2) + ((u ^ ((r >> 1) & 7)) << 4); }
  __device__ static __forceinline__ int b_lds_off(int r, int u) { return r * (BN * 2) + ((u ^ ((((r & 3) << 2) | (((r >> 3) & 1) << 1)) & (UB - 1))) << 4); }
  __device__ static __forceinline__ u32x4 load16(const unsigned char* p) {
    u32x4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 16);
    return v;
  }
};

// ---- an output tile on any 2-byte boundaries -----------------------------------------------------------------------------
// `width` values from column c of the tile's row r; the columns before col_first are another tile's (the last tile of a row is moved back into z).
template <typename OutT>
struct LooseOutput {
  OutT* z;
  int32_t ldz, row0, col0, col_first, cover_m, cover_n, accumulate;

  template <int W>
  __device__ __forceinline__ void store(int r, int c, const float* v) const {
    const int32_t gr = row0 + r, gc = col0 + c;
    if (gr >= cover_m || gc >= cover_n) return;
    OutT* dst = z + (int64_t)gr * ldz + gc;
    if (gc >= col_first && gc + W <= cover_n) {
      OutT o[W];
      if (accumulate) __builtin_memcpy(o, __builtin_assume_aligned(dst, sizeof(OutT)), sizeof(o));
#pragma unroll
      for (int e = 0; e < W; ++e) o[e] = (OutT)(accumulate ? v[e] + (float)o[e] : v[e]);
      __builtin_memcpy(__builtin_assume_aligned(dst, sizeof(OutT)), o, sizeof(o));
    } else {
#pragma unroll
      for (int e = 0; e < W; ++e)
        if (gc + e >= col_first && gc + e < cover_n) dst[e] = (OutT)(accumulate ? v[e] + (float)dst[e] : v[e]);
    }
  }
};
// A pass puts as many rows of the tile as fit into the stages as f32 (16-byte chunk c of row r at chunk c ^ (r & 15)), then a thread takes 8
// neighbouring columns of a row at a time: take(row, unit of 8 columns, the two halves).
template <int BM, int BN, int WM, int WN, int THREADS, int LDS_BYTES, int TN, int TM, typename F>
__device__ __forceinline__ void output_passes(const f32x4 (&acc)[TN][TM], unsigned char* lds, int wm, int wn, int32_t rows, F&& take) {
  constexpr int kOutRows = LDS_BYTES / (BN * 4) < BM ? LDS_BYTES / (BN * 4) : BM, kOutPasses = (BM + kOutRows - 1) / kOutRows, UB = BN / 8;
  static_assert(kOutRows % WM == 0 || WM % kOutRows == 0, "an output pass takes whole wavefront sub-tiles");
  const int tid = threadIdx.x, l16 = tid & 15, grp = (tid & 63) >> 4;
  for (int pass = 0; pass < kOutPasses; ++pass) {
    __syncthreads();   // the stages (or the previous pass) have been read
    const int first = pass * kOutRows;
    if (wm * WM < first + kOutRows && first < wm * WM + WM) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        const int r = wm * WM + tm * 16 + l16 - first;
        if (kOutPasses > 1 && (wm * WM + tm * 16 < first || wm * WM + tm * 16 >= first + kOutRows)) continue;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          *reinterpret_cast<f32x4*>(lds + r * (BN * 4) + (((wn * (WN / 4) + tn * 4 + grp) ^ (r & 15)) << 4)) = acc[tn][tm];
      }
    }
    __syncthreads();
    for (int o = tid; o < kOutRows * UB; o += THREADS) {
      const int r = o / UB, u = o % UB;
      if (first + r >= BM || first + r >= rows) break;   // rows only grow with o
      take(first + r, u, *reinterpret_cast<const f32x4*>(lds + r * (BN * 4) + (((2 * u) ^ (r & 15)) << 4)),
           *reinterpret_cast<const f32x4*>(lds + r * (BN * 4) + (((2 * u + 1) ^ (r & 15)) << 4)));
    }
  }
}

// ---- register-staged 256 x 256 tiles -------------------------------------------------------------------------------------------
// GemmStaged (gemm_small.hip) on 256 x 256: eight wavefronts of 128 x 64 outputs read 96 KiB of LDS for 2 MFLOP where those of 64 x 64 on 256 x 128 tiles read 128.  128 accumulators leave
// no room for two sets of fragments or two K tiles of loads: the x fragments are one set, each read again behind its last MFMA (as on the ring,
// gemm_ring16.h), and twelve 16-byte loads, one and a half K tiles, are in flight in a queue: a thread writes the oldest to the next stage and
// asks for another in its place.  One barrier per K tile, behind three of its four blocks of 16 MFMAs.  For
// outputs of 129 to 256 such tiles, two rounds of 256 x 128, and for a long K in many rounds: bf16 200 x 50021 x 1024 46.3 -> 37.3 us.
template <typename OutT, typename InT>
struct GemmStagedWide : StagedLayout<256> {
  static constexpr int BM = 256, BN = 256, kThreads = 512, WM = 128, WN = 64, TM = 8, TN = 4, TMH = 4;
  static constexpr int kABytes = BM * BK * 2, kStageBytes = kABytes + BK * BN * 2, kPieces = 8, kQueue = 12;

  __device__ static void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, int32_t k_total, int32_t cover_m, int32_t cover_n,
                             int32_t accumulate, uint32_t tiles_m, uint32_t tiles_n) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kStageBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / 4, wn = wave % 4, l16 = lane & 15, grp = lane >> 4;
    uint32_t pm, pn;
    grouped_tile(xcd_contiguous(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, &pm, &pn);
    const int32_t M = x.shape[0], N = y.shape[1];
    const int64_t lda = (int64_t)x.strides[0] * 2, ldb = (int64_t)y.strides[0] * 2;   // bytes
    const int32_t k_valid = min(min(x.shape[1], y.shape[0]), k_total), full = k_valid / BK;
    const int32_t row0 = pm * BM, col_first = pn * BN, col0 = max(0, min(col_first, N - BN));
    const int a_r = tid / 8, b_r = tid / UB, a_k = tid % 8 * 8;
    uint32_t a_off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a_off[i] = (uint32_t)(min(row0 + a_r + i * 64, M - 1) * lda) + a_k * 2;   // rows past the end repeat the last one
    const uint32_t b_off = (uint32_t)(b_r * ldb) + (uint32_t)(col0 + tid % UB * 8) * 2;
    const int a_st = a_lds_off(a_r, tid % 8), b_st = 2 * kABytes + b_lds_off(b_r, tid % UB);   // 64 rows of x and 16 of y further on the swizzle is the same
    const unsigned char* const xp = (const unsigned char*)x.ptr;
    const unsigned char* const yp = (const unsigned char*)y.ptr;
    // piece p of a K tile: 64 rows of x, then 16 K rows of y; nothing behind the last whole K tile.  Through descriptors (operands end below 2
    // GiB), a register and a scalar to an address: with 64-bit addresses the loop had no room for them.
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(xp, (uint32_t)((M - 1) * lda + x.shape[1] * 2)), ry = make_rsrc(yp, (uint32_t)((y.shape[0] - 1) * ldb + N * 2));
    const uint32_t y_step = (uint32_t)ldb;
    auto load = [&](int32_t kt, int p) {
      const uint32_t dead = kt < full ? 0u : 0x80000000u;
      return p < 4 ? __builtin_amdgcn_raw_buffer_load_b128(rx, a_off[p] | dead, kt * (BK * 2), 0)
                   : __builtin_amdgcn_raw_buffer_load_b128(ry, b_off | dead, (kt * BK + (p - 4) * 16) * y_step, 0);
    };
    auto write = [&](unsigned char* s, int p, u32x4 v) { *reinterpret_cast<u32x4*>(s + (p < 4 ? a_st + p * 8192 : b_st + (p - 4) * 8192)) = v; };

    const int tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
    int a_addr[2], b_addr[TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_addr[ks] = a_lds_off(wm * WM + l16, ks * 4 + grp);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = wn * WN + tn * 16 + tr_col;
      b_addr[tn] = 2 * kABytes + b_lds_off(grp * 8 + tr_row, n >> 3) + (n & 7) * 2;
    }
    auto read_a = [&](const unsigned char* s, int ks, int mh, bf16x8 (&into)[TMH], int i) {
      into[i] = *reinterpret_cast<const bf16x8*>(s + a_addr[ks] + (mh * TMH + i) * (16 * BK * 2));
    };
    auto read_b = [&](const unsigned char* s, int ks, bf16x8 (&into)[TN], int tn) {
      const unsigned char* p = s + b_addr[tn] + ks * 32 * (BN * 2);
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 4 * (BN * 2)));
      into[tn] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // both x stages, then both y stages: an address and a 16-bit immediate reach either
    unsigned char* const s0 = lds;
    unsigned char* const s1 = lds + kABytes;
    u32x4 q[kQueue];
    bf16x8 af[TMH], b0[TN], b1[TN];
    // rows [mh * 64, ..) of the sub-tile by its columns; between the MFMAs the next block's x fragments, the next K step's y fragments (`ib`,
    // where rd_y) and the queue's pieces first .. last - 1 of K tile kt + 1, of which piece 0 lies at `head`
    auto block = [&](const bf16x8 (&ub)[TN], int mh, const unsigned char* rd, int rd_ks, int rd_mh, bool rd_y, bf16x8 (&ib)[TN], unsigned char* to, int32_t kt,
                     auto head, int first, int last) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int tm = j / TN, tn = j % TN;
        if (rd_y && j % 4 == 0) read_b(rd, rd_ks, ib, j / 4);
#pragma unroll
        for (int p = 0; p < kPieces; ++p)
          if (p >= first && p < last && (p - first) * 16 / (last - first) + 1 == j) {
            u32x4& slot = q[(decltype(head)::value + p) % kQueue];
            write(to, p, slot);
            slot = load(kt + (p < 4 ? 2 : 3), (p + 4) % kPieces);
          }
        acc[tn][mh * TMH + tm] = mfma_16x16x32<InT>(ub[tn], af[tm], acc[tn][mh * TMH + tm]);
        if (tn == TN - 1) read_a(rd, rd_ks, rd_mh, af, tm);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto k_tile = [&](unsigned char* cur, unsigned char* next, int32_t kt, auto head) {
      block(b0, 0, cur, 0, 1, false, b1, next, kt, head, 0, 3);
      block(b0, 1, cur, 1, 0, true, b1, next, kt, head, 3, 5);
      block(b1, 0, cur, 1, 1, false, b0, next, kt, head, 5, 8);
      __syncthreads();   // tile kt + 1 is whole, and tile kt in registers everywhere
      block(b1, 1, next, 0, 0, true, b0, next, kt, head, 0, 0);
    };
    if (full > 0) {
#pragma unroll
      for (int p = 0; p < kQueue; ++p) q[p] = load(p / kPieces, p % kPieces);
#pragma unroll
      for (int p = 0; p < kPieces; ++p) {
        write(s0, p, q[p]);
        q[p] = load((p + kQueue) / kPieces, (p + kQueue) % kPieces);
      }
      __syncthreads();
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) read_b(s0, 0, b0, tn);
#pragma unroll
      for (int i = 0; i < TMH; ++i) read_a(s0, 0, 0, af, i);
    }
    // (the queue's head and the stages come round every six K tiles; behind the last one nothing is read that was written)
#pragma unroll 1
    for (int32_t kt = 0; kt < full; kt += 6) {
      k_tile(s0, s1, kt, std::integral_constant<int, 8>{});
      if (kt + 1 >= full) break;
      k_tile(s1, s0, kt + 1, std::integral_constant<int, 4>{});
      if (kt + 2 >= full) break;
      k_tile(s0, s1, kt + 2, std::integral_constant<int, 0>{});
      if (kt + 3 >= full) break;
      k_tile(s1, s0, kt + 3, std::integral_constant<int, 8>{});
      if (kt + 4 >= full) break;
      k_tile(s0, s1, kt + 4, std::integral_constant<int, 4>{});
      if (kt + 5 >= full) break;
      k_tile(s1, s0, kt + 5, std::integral_constant<int, 0>{});
    }

    // The ragged last K tile, straight into a stage: K positions past the end are 0 on both sides.
    if (k_valid % BK != 0) {
      const int32_t k0 = full * BK;
      __syncthreads();
#pragma unroll 1
      for (int c = tid; c < BM * 8; c += kThreads) {
        const int32_t k = k0 + c % 8 * 8;
        const unsigned char* row = xp + (int64_t)min(row0 + c / 8, M - 1) * lda;
        u32x4 v = {0, 0, 0, 0};
        if (k + 8 <= k_valid) {
          v = load16(row + (int64_t)k * 2);
        } else if (k < k_valid) {
          uint32_t h[4] = {0, 0, 0, 0};
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (k + e < k_valid) h[e / 2] |= (uint32_t)reinterpret_cast<const uint16_t*>(row)[k + e] << (e % 2 * 16);
          v = u32x4{h[0], h[1], h[2], h[3]};
        }
        *reinterpret_cast<u32x4*>(s0 + a_lds_off(c / 8, c % 8)) = v;
      }
#pragma unroll 1
      for (int c = tid; c < BK * UB; c += kThreads) {
        const int32_t k = k0 + c / UB;
        u32x4 v = {0, 0, 0, 0};
        if (k < k_valid) v = load16(yp + k * ldb + (int64_t)(col0 + c % UB * 8) * 2);
        *reinterpret_cast<u32x4*>(s0 + 2 * kABytes + b_lds_off(c / UB, c % UB)) = v;
      }
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) read_b(s0, ks, b0, tn);
#pragma unroll
        for (int mh = 0; mh < 2; ++mh) {
#pragma unroll
          for (int i = 0; i < TMH; ++i) read_a(s0, ks, mh, af, i);
#pragma unroll
          for (int i = 0; i < TMH; ++i)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) acc[tn][mh * TMH + i] = mfma_16x16x32<InT>(b0[tn], af[i], acc[tn][mh * TMH + i]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    const LooseOutput<OutT> out{(OutT*)z.ptr, z.strides[0], row0, col0, col_first, cover_m, cover_n, accumulate};
    output_passes<BM, BN, WM, WN, kThreads, 2 * kStageBytes>(acc, lds, wm, wn, cover_m - row0, [&](int r, int u, f32x4 lo, f32x4 hi) {
      const float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      out.template store<8>(r, u * 8, f);
    });
  }
};

}  // namespace gemm
}  // namespace cutile

#define GEMM_STAGED_WIDE_KERNEL(NAME, IN_T, OUT_T)                                                                                  \
  extern "C" __global__ void __launch_bounds__(512, 2)                                                                              \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k_total, int32_t cover_m, int32_t cover_n,       \
                         int32_t accumulate, float*, uint32_t*, uint32_t tiles_m, uint32_t tiles_n, uint32_t) {                      \
    GemmStagedWide<OUT_T, IN_T>::run(z, x, y, k_total, cover_m, cover_n, accumulate, tiles_m, tiles_n);                              \
  }
