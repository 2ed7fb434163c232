// GEMM tiles between 128 x 128 and 256 x 256, for outputs that 256 x 256 tiles do not fill the chip with.  The K tiles of an output tile
// may be shared by several workgroups (split_k.h); the rule that picks tile and split is ring_plan (host/gemm_choice.h).
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_common.h"
#include "gemm_ring16.h"
#include "kernel_args.h"
#include "split_k.h"

namespace cutile {
namespace gemm {

// ---- small tiles: whole stages, four or five of them ------------------------------------------------------------------------
// On tiles of 192 x 128 and less a K tile is 0.2 to 0.3 us of matrix work, and the ring of three x and two y stages (gemm_ring16.h) is
// bound by the wait in front of each of its two barriers per K tile: every LDS read has to be home, and the y half behind it was
// requested 1.25 K tiles ago, less than a fetch that misses L2 takes.  LDS holds four (192 x 128) or five (128 x 128) whole stages of
// such a tile.  Tile kt + STAGES - 1 goes into the stage that tile kt - 1 left, behind the one barrier in the middle of tile kt: by then
// every wavefront has multiplied with its last fragment of tile kt - 1, so nothing needs to be waited for but the fetches of tile
// kt + 1, requested STAGES - 2 K tiles ago.  Fragments are double-buffered (a K step of 32 is read while the one before it is
// multiplied), and eight wavefronts, two to a SIMD, keep the matrix pipe fed across each other's waits (four of them: 178 us where eight
// take 164 at 1500 x 4096 x 14336).
// f16, us on the ring and here, operands from memory (and from the caches): 1500 x 4096 x 14336, 256 tiles of 192 x 128, 189 and 169 (181, 157);
// 1500 x 4096 x 4096 57.7 and 52.1 (54.7, 48.8); on 128 x 128 tiles 1500 x 1024 x 4096, 96 of them, here with K shared by two, 38.6 and 25.5 (35.3,
// 23.8), 2048 x 2048 x 2048, 256 of them, 24.1 and 22.9.
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, typename InT>
struct GemmStages {
  static constexpr int BK = 64, kWaves = WAVES_M * WAVES_N, kThreads = kWaves * 64;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 16, TN = WN / 16, NB = TM * TN;
  static constexpr int UB = BN / 8;                                      // 16-byte units of a y-tile row
  static constexpr int kAInstr = BM / 8 / kWaves, kBRows = 64 / UB, kBInstr = BK / kBRows / kWaves, kFetch = kAInstr + kBInstr;
  static constexpr int kABytes = BM * BK * 2, kStageBytes = kABytes + BK * BN * 2;
  static_assert(BM % (8 * kWaves) == 0 && BK % (kBRows * kWaves) == 0 && UB >= 16 && UB <= 64, "tile must split evenly");
  static_assert(TM % 2 == 0, "the epilogue takes 32-row bands");
  static_assert((STAGES == 4 || STAGES == 5) && STAGES * kStageBytes <= 160 * 1024, "the stages must fit LDS");

  __device__ static __forceinline__ int a_lds_off(int r, int u) { return r * (BK * 2) + ((u ^ ((r >> 1) & 7)) << 4); }
  __device__ static __forceinline__ int b_swizzle(int r) { return ((r & 3) << 2) | (((r >> 3) & 1) << 1); }
  __device__ static __forceinline__ int b_lds_off(int r, int u) { return r * (BN * 2) + ((u ^ b_swizzle(r)) << 4); }
  static constexpr int wait_vm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }   // vmcnt(n) alone

  __device__ static __forceinline__ void run(const PartitionArg<2>& z, TensorArg<2> x, TensorArg<2> y, int32_t k_total,
                                             const TileGrid& g, int32_t accumulate, float* partials, uint32_t* counters, uint32_t splits) {
    __shared__ __attribute__((aligned(1024))) unsigned char st0[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st1[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st2[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st3[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st4[STAGES > 4 ? kStageBytes : 16];
    const SplitTile t = split_tile<BK, 2>(g.x, g.y, splits, x, y, k_total);
    const uint32_t pm = t.pm, pn = t.pn;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int32_t M = x.shape[0], N = y.shape[1], lda = x.strides[0], ldb = y.strides[0];
    const int32_t row0 = pm * BM, col0 = pn * BN;
    const int32_t k_valid = min(min(x.shape[1], y.shape[0]), k_total);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(x.ptr, (uint32_t)(((int64_t)(M - 1) * lda + x.shape[1]) * 2));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(y.ptr, y.shape[0] > 0 ? (uint32_t)(((int64_t)(y.shape[0] - 1) * ldb + N) * 2) : 0u);
    constexpr uint32_t kOob = 0x80000000u;
    uint32_t a_goff[kAInstr], b_goff[kBInstr];
    int32_t a_klim[kAInstr];
    const int32_t b_klim = k_valid - (int32_t)(lane / UB);
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) {
      const int r = (wave * kAInstr + i) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
      a_goff[i] = row0 + r < M ? (uint32_t)(((int64_t)(row0 + r) * lda + u * 8) * 2) : kOob;
      a_klim[i] = k_valid - u * 8;
    }
#pragma unroll
    for (int i = 0; i < kBInstr; ++i) {
      const int r = (i * kWaves + wave) * kBRows + lane / UB, u = (lane % UB) ^ b_swizzle(r);
      b_goff[i] = col0 + u * 8 < N ? (uint32_t)(((int64_t)r * ldb + col0 + u * 8) * 2) : kOob;
    }
    auto fetch = [&](unsigned char* stage, int32_t k0, int i) {
      if (i < kAInstr)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_PTR(void))(stage + (wave * kAInstr + i) * 1024), 16, k0 < a_klim[i] ? a_goff[i] : kOob, k0 * 2, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LDS_PTR(void))(stage + kABytes + ((i - kAInstr) * kWaves + wave) * 1024), 16,
                                                 k0 + ((i - kAInstr) * kWaves + wave) * kBRows < b_klim ? b_goff[i - kAInstr] : kOob, k0 * ldb * 2, 0, 0);
    };

    const int grp = lane >> 4, l16 = lane & 15, tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
    int a_addr[2], b_addr[TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_addr[ks] = a_lds_off(wm * WM + l16, ks * 4 + grp);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = wn * WN + tn * 16 + tr_col;
      b_addr[tn] = kABytes + b_lds_off(grp * 8 + tr_row, n >> 3) + (n & 7) * 2;
    }
    struct Frags {
      bf16x8 a[TM], b[TN];
    };
    // unit i of a K step's operands: the y fragments and the first x fragment are needed first
    auto read = [&](const unsigned char* stage, int ks, Frags& f, int i) {
      if (i < TN) {
        const unsigned char* p = stage + b_addr[i] + ks * 32 * (BN * 2);
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
        s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 4 * (BN * 2)));
        f.b[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      } else {
        f.a[i - TN] = *reinterpret_cast<const bf16x8*>(stage + a_addr[ks] + (i - TN) * (16 * BK * 2));
      }
    };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    constexpr int UNITS = TM + TN;
    auto step = [&](const Frags& f, Frags& next, const unsigned char* rd, int rd_ks, bool fill, unsigned char* fill_stage, int32_t fill_k0) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
#pragma unroll
        for (int i = 0; i < UNITS; ++i)
          if (i * (NB - 2) / UNITS == j) read(rd, rd_ks, next, i);
        if (fill) {
#pragma unroll
          for (int i = 0; i < kFetch; ++i)
            if (i * NB / kFetch == j) fetch(fill_stage, fill_k0, i);
        }
        acc[j % TN][j / TN] = mfma_16x16x32<InT>(f.b[j % TN], f.a[j / TN], acc[j % TN][j / TN]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    const int32_t k_tiles = (k_total + BK - 1) / BK;
    Frags f0, f1;
    auto fetch_tile = [&](unsigned char* stage, int32_t kt) {
#pragma unroll
      for (int i = 0; i < kFetch; ++i) fetch(stage, kt * BK, i);
    };
    fetch_tile(st0, 0);
    fetch_tile(st1, 1);
    fetch_tile(st2, 2);
    if (STAGES > 4) fetch_tile(st3, 3);
    __builtin_amdgcn_s_waitcnt(wait_vm((STAGES - 2) * kFetch));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < UNITS; ++i) read(st0, 0, f0, i);

    auto k_tile = [&](unsigned char* cur, const unsigned char* next, unsigned char* prev, int32_t kt) {
      step(f0, f1, cur, 1, false, prev, 0);
      __builtin_amdgcn_s_waitcnt(wait_vm((STAGES - 3) * kFetch));
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      step(f1, f0, next, 0, true, prev, (kt + STAGES - 1) * BK);
    };
    int32_t kt = 0;
    if constexpr (STAGES == 4) {
      for (; kt + 4 <= k_tiles; kt += 4) {
        k_tile(st0, st1, st3, kt);
        k_tile(st1, st2, st0, kt + 1);
        k_tile(st2, st3, st1, kt + 2);
        k_tile(st3, st0, st2, kt + 3);
      }
      if (kt < k_tiles) k_tile(st0, st1, st3, kt);
      if (kt + 1 < k_tiles) k_tile(st1, st2, st0, kt + 1);
      if (kt + 2 < k_tiles) k_tile(st2, st3, st1, kt + 2);
    } else {
      for (; kt + 5 <= k_tiles; kt += 5) {
        k_tile(st0, st1, st4, kt);
        k_tile(st1, st2, st0, kt + 1);
        k_tile(st2, st3, st1, kt + 2);
        k_tile(st3, st4, st2, kt + 3);
        k_tile(st4, st0, st3, kt + 4);
      }
      if (kt < k_tiles) k_tile(st0, st1, st4, kt);
      if (kt + 1 < k_tiles) k_tile(st1, st2, st0, kt + 1);
      if (kt + 2 < k_tiles) k_tile(st2, st3, st1, kt + 2);
      if (kt + 3 < k_tiles) k_tile(st3, st4, st2, kt + 3);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (splits > 1 && !combine_tile<TM, TN, kThreads>(acc, partials + (size_t)t.tile * splits * (BM * BN), counters + t.tile, t.split, splits, reinterpret_cast<uint32_t*>(st2))) return;   // (no output band lies in stage 2)
    constexpr int PER = kStageBytes / kEpilogueBytesPerWave<WN>;
    static_assert(kWaves <= 2 * PER, "the output bands must fit the stages");
    unsigned char* band = (wave < PER ? st0 : st1) + wave % PER * kEpilogueBytesPerWave<WN>;
    store_tile_staged16<TM, TN, InT>(acc, band, (InT*)z.ptr, z.strides[0], z.shape[0], z.shape[1], row0 + wm * WM, col0 + wn * WN, lane, accumulate);
  }
};

}  // namespace gemm
}  // namespace cutile

#define GEMM_STAGES_KERNEL(NAME, BM, BN, WVM, WVN, STAGES, T)                                                                        \
  extern "C" __global__ void __launch_bounds__(WVM * WVN * 64)                                                                      \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k, TileGrid g, int32_t accumulate,               \
                         float* partials, uint32_t* counters, uint32_t splits) {                                                    \
    GemmStages<BM, BN, WVM, WVN, STAGES, T>::run(z, x, y, k, g, accumulate, partials, counters, splits);                            \
  }
#define GEMM_RING_TILE_KERNEL(NAME, BM, BN, WVM, WVN, T)                                                                                  \
  extern "C" __global__ void __launch_bounds__(WVM * WVN * 64)                                                                      \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k, TileGrid g, int32_t accumulate,               \
                         float* partials, uint32_t* counters, uint32_t splits) {                                                    \
    using Ring = GemmRing16<BM, BN, WVM, WVN, T, T>;                                                                                \
    const SplitTile t = split_tile<64, 2>(g.x, g.y, splits, x, y, k);                                                                \
    Ring::run_tile(z, x, y, k, t.pm, t.pn, accumulate, [&](auto& acc, uint32_t* flag) {                                              \
      return splits == 1 || combine_tile<Ring::TM, Ring::TN, Ring::kThreads>(acc, partials + (size_t)t.tile * splits * (BM * BN),     \
                                                                             counters + t.tile, t.split, splits, flag);             \
    });                                                                                                                             \
  }

// Tiles of two widths in one launch: `wide` columns of BM x 256 tiles, then columns of BM x 192, in the stages of the former.  Outputs of one and a half to two
// rounds of workgroups leave compute units idle in the second; with the widths mixed every compute unit has about as much to do.  f16, us on
// one width and on two: 1344 x 12032 x 4608 161, 152; 900 x 18432 x 5120 179, 172; 560 x 28672 x 4096 148, 141; 1700 x 11000 x 2048 79.6, 76.8.  Least
// where idle units had given the others clock (1.93 GHz with two widths, below the chip's 2.4): 1500 x 14336 x 4096 161.7, 160.9, in a block over a prompt of
// 1500 167.3, 163.7.  400 drawn products of one to two rounds take 0.995 of the time before, at most 1.035 (within what the card varies).
#define GEMM_RING_MIX_KERNEL(NAME, BM, T)                                                                                           \
  extern "C" __global__ void __launch_bounds__(512)                                                                                 \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k, TileGrid g, int32_t accumulate,               \
                         float*, uint32_t*, uint32_t narrow) {                                                                      \
    using Wide = GemmRing16<BM, 256, 2, 4, T, T>;                                                                                   \
    using Narrow = GemmRing16<BM, 256, 2, 4, T, T, 192>;                                                                            \
    __shared__ __attribute__((aligned(1024))) unsigned char xs0[Wide::kABytes];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char xs1[Wide::kABytes];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char xs2[Wide::kABytes];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char ys0a[Wide::kBBytes / 2];                                                \
    __shared__ __attribute__((aligned(1024))) unsigned char ys0b[Wide::kBBytes / 2];                                                \
    __shared__ __attribute__((aligned(1024))) unsigned char ys1a[Wide::kBBytes / 2];                                                \
    __shared__ __attribute__((aligned(1024))) unsigned char ys1b[Wide::kBBytes / 2];                                                \
    const uint32_t first = g.x * g.y;                                                                                               \
    uint32_t pm, pn;                                                                                                                \
    if (blockIdx.x < first) {                                                                                                       \
      grouped_tile(xcd_contiguous(blockIdx.x, first), g.x, g.y, &pm, &pn);                                                          \
      Wide::run_tile_in({xs0, xs1, xs2, ys0a, ys0b, ys1a, ys1b}, z, x, y, k, pm, pn, accumulate);                                   \
    } else {                                                                                                                        \
      grouped_tile(xcd_contiguous(blockIdx.x - first, g.x * narrow), g.x, narrow, &pm, &pn);                                        \
      const int32_t at = (int32_t)g.y * 256;                                                                                        \
      y.ptr = (T*)y.ptr + at, y.shape[1] -= at;                                                                                     \
      z.ptr = (T*)z.ptr + at, z.shape[1] -= at;                                                                                     \
      Narrow::run_tile_in({xs0, xs1, xs2, ys0a, ys0b, ys1a, ys1b}, z, x, y, k, pm, pn, accumulate);                                 \
    }                                                                                                                               \
  }
