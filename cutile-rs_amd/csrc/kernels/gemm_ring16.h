// The ring-pipelined GEMM tile body on v_mfma_f32_16x16x32 (gemm_bf16.hip, gemm_small.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_common.h"
#include "mapped_partition.h"
#include "kernel_args.h"

namespace cutile {
namespace gemm {

// ---- the ring variant on v_mfma_f32_16x16x32 -----------------------------------------------
// Same stages, fetches, barriers and wait counts as GemmRing; the matrix instruction is the 16 x 16 x 32 form.
// On this chip the matrix kernels run against the power limit, and per flop the 16 x 16 x 32 form writes half as
// many accumulator values as 32 x 32 x 16: a loop of nothing but MFMAs on random bf16 operands sustains
// 2093 TFLOP/s with it against 1854 (equal, 2463 - 2481, on constant operands).  A block is 16 MFMAs (half of the
// sub-tile's rows by all of its columns, one 32-wide K step) and lasts as long as a block of GemmRing; the y
// fragments of a K step serve two blocks, so LDS traffic is unchanged.
// CN < BN: the stages of a BN-column tile hold CN columns (of a tile beside wider ones, gemm_tiles.h); fetches of the others bring nothing.
template <int BM, int BN, int WAVES_M, int WAVES_N, typename OutT, typename InT = __bf16, int CN = BN>
struct GemmRing16 {
  static constexpr int BK = 64;
  static constexpr int kWaves = WAVES_M * WAVES_N;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int WM = BM / WAVES_M, WN = CN / WAVES_N, BAND = BN / WAVES_N;   // BAND: columns that a row of an output band has room for
  static constexpr int TM = WM / 16, TN = WN / 16;   // 16 x 16 accumulator blocks of the wavefront's sub-tile
  static constexpr int TMH = TM / 2;                   // x fragments of one MFMA block (half the sub-tile's rows)
  static_assert(TM % 2 == 0, "a block takes half of the sub-tile's rows");
  static constexpr int UB = BN / 8;                         // 16-byte units per y-tile row
  static constexpr int kAInstr = BM / 8 / kWaves;           // 1 KiB = 8 x-tile rows
  static constexpr int kBRowsPerInstr = 64 / UB;
  static constexpr int kBInstr = BK / kBRowsPerInstr / kWaves;
  static constexpr int kABytes = BM * BK * 2, kBBytes = BK * BN * 2;
  static constexpr int kLdsBytes = 3 * kABytes + 2 * kBBytes;
  static_assert(BM % (8 * kWaves) == 0 && BK % (kBRowsPerInstr * kWaves) == 0, "tile must split evenly");
  static_assert(UB >= 16 && UB <= 64, "y-tile row must be 16..64 units");
  static_assert(kBInstr % 2 == 0, "each wavefront fetches the same share of both y halves");
  static_assert(kAInstr + kBInstr <= 15, "the wait count must fit the low vmcnt field");

  __device__ static __forceinline__ int a_lds_off(int r, int u) { return r * (BK * 2) + ((u ^ ((r >> 1) & 7)) << 4); }
  // y rows 8 apart are read by neighbouring lane groups of one transposing read: bit 3 of the row moves them 32 bytes apart
  __device__ static __forceinline__ int b_swizzle(int r) { return ((r & 3) << 2) | (((r >> 3) & 1) << 1); }
  __device__ static __forceinline__ int b_lds_off(int r, int u) { return r * (BN * 2) + ((u ^ b_swizzle(r)) << 4); }


  __device__ static void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y,
                             int32_t k_total, const TileGrid& g, int32_t accumulate) {
    // One K tile, or two of a large output, read little against what is written: the plain order where the tiles are no multiple of 8 (us in the
    // contiguous order and in this one, f16: 4794 x 10880 x 64, 817 tiles, 34.8, 34.2, accumulating 53.4, 50.9; 7725 x 11392 x 64 48.1, 46.9 and 82.3,
    // 79.5; bf16 7804 x 12480 x 128, 1519 tiles, 59.0, 57.2; 6654 x 8704 x 128 38.9, 38.1).  Two K tiles of fewer tiles, and longer K, are read
    // faster in the contiguous order (2967 x 8768 x 128, 420 tiles, 21.6, 22.4; 3557 x 14912 x 256 48.8, 50.8).
    uint32_t pm, pn;
    if (g.x * g.y % kNumXcd != 0 && (k_total <= BK || (k_total <= 2 * BK && g.x * g.y > 512)))
      grouped_tile(blockIdx.x, g.x, g.y, &pm, &pn);
    else
      tile_coords(g.x, g.y, &pm, &pn);
    run_tile(z, x, y, k_total, pm, pn, accumulate);
  }

  // gemm_persistent: workgroup b computes the tiles of stream items b, b + gridDim.x, ... of the mapped output
  // partition from zero accumulators, in the XCD-contiguous order of GemmDirect::run_persistent.
  __device__ static void run_persistent(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y,
                                        const MappedArg& m) {
    for (uint32_t item = blockIdx.x; item < m.total; item += gridDim.x) {
      const uint32_t pos = m.total % kNumXcd == 0 ? (item % kNumXcd) * (m.total / kNumXcd) + item / kNumXcd : item;
      uint32_t bid[3];
      mapped_index(m, pos, bid);
      run_tile(z, x, y, x.shape[1], bid[0], bid[1], 0);
      __syncthreads();   // the output bands live in the stages that the next tile refills
    }
  }

  // gemm launched with one workgroup per compute unit ("p"): workgroup b walks the tiles b, b + gridDim.x, ... of the
  // launch's XCD-contiguous, M-grouped order, tile after tile with the full tile body (any extents, any K, z as the
  // initial accumulator or not).  Against one workgroup per tile it saves the workgroup starts and keeps each XCD on
  // one contiguous eighth of the order round by round.
  __device__ static void run_walk(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, int32_t k_total,
                                  const TileGrid& g, int32_t accumulate) {
    const uint32_t total = g.x * g.y;
    for (uint32_t item = blockIdx.x; item < total; item += gridDim.x) {
      uint32_t pm, pn;
      tile_of_id(item, g.x, g.y, gridDim.x, &pm, &pn);
      run_tile(z, x, y, k_total, pm, pn, accumulate);
      __syncthreads();   // the output bands live in the stages that the next tile refills
    }
  }

  struct Stages {
    unsigned char *xs0, *xs1, *xs2, *ys0a, *ys0b, *ys1a, *ys1b;
  };
  struct AllOfK {
    template <typename Acc>
    __device__ __forceinline__ bool operator()(Acc&, uint32_t*) const { return true; }
  };
  // `combine(acc, flag)`: adds what other workgroups have summed of this tile; false where another one stores it
  template <typename Combine = AllOfK>
  __device__ static __forceinline__ void run_tile(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y,
                                                  int32_t k_total, uint32_t pm, uint32_t pn, int32_t accumulate, Combine combine = Combine{}) {
    // Separately named stages: the compiler can then tell a refill of one from
    // operand reads of another and adds no waits of its own.
    __shared__ __attribute__((aligned(1024))) unsigned char xs0[kABytes];
    __shared__ __attribute__((aligned(1024))) unsigned char xs1[kABytes];
    __shared__ __attribute__((aligned(1024))) unsigned char xs2[kABytes];
    __shared__ __attribute__((aligned(1024))) unsigned char ys0a[kBBytes / 2];  // y stage 0, K rows 0..31
    __shared__ __attribute__((aligned(1024))) unsigned char ys0b[kBBytes / 2];  //            K rows 32..63
    __shared__ __attribute__((aligned(1024))) unsigned char ys1a[kBBytes / 2];
    __shared__ __attribute__((aligned(1024))) unsigned char ys1b[kBBytes / 2];
    run_tile_in(Stages{xs0, xs1, xs2, ys0a, ys0b, ys1a, ys1b}, z, x, y, k_total, pm, pn, accumulate, combine);
  }
  template <typename Combine = AllOfK>
  __device__ static __forceinline__ void run_tile_in(const Stages& stages, const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y,
                                                     int32_t k_total, uint32_t pm, uint32_t pn, int32_t accumulate, Combine combine = Combine{}) {
    unsigned char *const xs0 = stages.xs0, *const xs1 = stages.xs1, *const xs2 = stages.xs2;
    unsigned char *const ys0a = stages.ys0a, *const ys0b = stages.ys0b, *const ys1a = stages.ys1a, *const ys1b = stages.ys1b;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int32_t M = x.shape[0], N = y.shape[1];
    const int32_t lda = x.strides[0], ldb = y.strides[0];
    const int32_t row0 = pm * BM, col0 = pn * CN;
    const int32_t k_valid = min(min(x.shape[1], y.shape[0]), k_total);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(x.ptr, (uint32_t)(((int64_t)(M - 1) * lda + x.shape[1]) * 2));
    // (a group of inner size 0 has no row of y: the prologue's masked fetches must still find themselves out of range)
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(y.ptr, y.shape[0] > 0 ? (uint32_t)(((int64_t)(y.shape[0] - 1) * ldb + N) * 2) : 0u);
    constexpr uint32_t kOob = 0x80000000u;

    // Global side of the fetches (per lane, K tile 0; the K advance is scalar).
    // y instruction i of this wavefront covers K rows of half i / (kBInstr/2).
    // A lane fetches K positions k0 + 8 u .. + 7 of an x row and K row k0 + r of y: past the end of K (a ragged last
    // tile, or a trailing fetch beyond the last one) its offset is out of range and the fetch brings zeros.  K is a
    // multiple of 8, so a 16-byte unit is wholly inside K or wholly beyond it.
    uint32_t a_goff[kAInstr], b_goff[kBInstr];
    int32_t a_klim[kAInstr];      // k0 < a_klim[i]  <=>  the lane's unit of instruction i lies inside K
    const int32_t b_klim = k_valid - (int32_t)(lane / UB);   // k0 + (first row of the instruction) < b_klim  <=>  the lane's row does
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) {
      const int r = (wave * kAInstr + i) * 8 + (lane >> 3);
      const int u = (lane & 7) ^ ((r >> 1) & 7);
      a_goff[i] = (row0 + r < M) ? (uint32_t)(((int64_t)(row0 + r) * lda + u * 8) * 2) : kOob;
      a_klim[i] = k_valid - u * 8;
    }
#pragma unroll
    for (int i = 0; i < kBInstr; ++i) {
      const int r = (i * kWaves + wave) * kBRowsPerInstr + lane / UB;
      const int u = (lane % UB) ^ b_swizzle(r);
      b_goff[i] = (u * 8 < CN && col0 + u * 8 < N) ? (uint32_t)(((int64_t)r * ldb + col0 + u * 8) * 2) : kOob;
    }
    auto fetch_a = [&](unsigned char* stage, int32_t k0, int i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_PTR(void))(stage + (wave * kAInstr + i) * 1024), 16,
                                               k0 < a_klim[i] ? a_goff[i] : kOob, k0 * 2, 0, 0);
    };
    // `half` = the y half-stage receiving K rows 32*h..32*h+31, h = i / (kBInstr/2)
    auto fetch_b = [&](unsigned char* half, int32_t k0, int i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LDS_PTR(void))(half + ((i % (kBInstr / 2)) * kWaves + wave) * 1024),
                                               16, k0 + (i * kWaves + wave) * kBRowsPerInstr < b_klim ? b_goff[i] : kOob,
                                               k0 * ldb * 2, 0, 0);
    };

    // LDS side of the operand reads (byte offsets inside a stage).  v_mfma_f32_16x16x32: a lane holds 8 consecutive K
    // values (group lane / 16 of the 32-wide K step) of row lane % 16 of its operand.
    const int grp = lane >> 4, l16 = lane & 15;
    const int tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
    // x: the swizzle term of row r + 16 tm is that of row r, so one address per K step serves all row blocks
    // (16 rows = 16 * BK * 2 bytes further on, an immediate offset of the read)
    int a_addr[2], b_addr[TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_addr[ks] = a_lds_off(wm * WM + l16, ks * 4 + grp);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = wn * WN + tn * 16 + tr_col;
      const int kr = grp * 8 + tr_row;         // row inside the y half-stage that holds this K step; the swizzle of kr + 4 is the same
      b_addr[tn] = b_lds_off(kr, n >> 3) + (n & 7) * 2;
    }
    constexpr int NB = TMH * TN;  // MFMAs per block: half the sub-tile's rows, one 32-wide K step
    // x fragments i of rows [mh * TMH * 16, ..) at K step ks of stage xs
    auto read_a = [&](const unsigned char* xs, int ks, int mh, bf16x8 (&into)[TMH], int i) {
      into[i] = *reinterpret_cast<const bf16x8*>(xs + a_addr[ks] + (mh * TMH + i) * (16 * BK * 2));
    };
    // y fragment tn of the K step held by the half-stage yh
    auto read_b = [&](const unsigned char* yh, bf16x8 (&into)[TN], int tn) {
      const unsigned char* p = yh + b_addr[tn];
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 4 * (BN * 2)));
      into[tn] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    f32x4 acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[tn][tm][v] = 0.0f;

    // One MFMA block: rows [mh * TMH * 16, ..) of the sub-tile times all its columns, on the x fragments `a` and the
    // y fragments `ub`, row block by row block.  Dealt out between its MFMAs in this
    // order: refill instructions first..last of the x stage `fill_x` (if any) and of the y stage `fill_y`
    // (instructions fb0..fb1-1), then, if rd_y, the reads of the next K step's y fragments into `ib`.  The x
    // fragments are one set: as soon as the last MFMA on a row block has issued, its fragment is read again for the
    // next block (rd_x, rd_ks, rd_mh) — three row blocks of MFMAs before it is used.  A wavefront issues in order
    // and an MFMA holds the issue slot until the matrix pipe takes it, so memory work placed after a run of MFMAs
    // would start late; sched_barrier(0) after every step keeps the order written here.
    constexpr int SLOTS = NB;   // memory instructions spread over all the block's MFMAs: one per MFMA at most (measured +3 % over the first half only)
    // (what a block does besides its MFMAs is said by the flags with_y / with_fill_x and the range fb0..fb1: a null
    // test of an LDS pointer is a run-time test, address 0 being a valid one)
    auto block = [&](bf16x8 (&a)[TMH], const bf16x8 (&ub)[TN], int mh, const unsigned char* rd_x, int rd_ks, int rd_mh,
                     bool with_y, const unsigned char* rd_y, bf16x8 (&ib)[TN], bool with_fill_x, unsigned char* fill_x,
                     unsigned char* fill_y, int fb0, int fb1, int32_t k0_x, int32_t k0_y) {
      const int n_fill = (with_fill_x ? kAInstr : 0) + (fb1 - fb0);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int tm = j / TN, tn = j % TN;
#pragma unroll
        for (int i = 0; i < kAInstr + kBInstr; ++i) {
          if (i < n_fill && i * SLOTS / n_fill == j) {
            if (with_fill_x && i < kAInstr)
              fetch_a(fill_x, k0_x, i);
            else
              fetch_b(fill_y, k0_y, fb0 + i - (with_fill_x ? kAInstr : 0));
          }
        }
        if (with_y) {
#pragma unroll
          for (int q = 0; q < TN; ++q)
            if (q * SLOTS / TN == j) read_b(rd_y, ib, q);
        }
        acc[tn][mh * TMH + tm] = mfma_16x16x32<InT>(ub[tn], a[tm], acc[tn][mh * TMH + tm]);
        if (tn == TN - 1) read_a(rd_x, rd_ks, rd_mh, a, tm);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // s_waitcnt immediate of gfx9: vmcnt [3:0] (and [15:14]), expcnt [6:4], lgkmcnt [11:8].
    constexpr int kWaitOlderLoads = (kAInstr + kBInstr) | (7 << 4) | (0 << 8);
    constexpr int kWaitPrologue = ((2 * kAInstr + 3 * kBInstr / 2) & 15) | (7 << 4) | (0 << 8) | (((2 * kAInstr + 3 * kBInstr / 2) >> 4) << 14);

    const int k_tiles = (k_total + BK - 1) / BK;
    bf16x8 af[TMH], b0[TN], b1[TN];
    // Prologue, in the issue order the steady state would have produced.
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) fetch_a(xs0, 0, i);
#pragma unroll
    for (int i = 0; i < kBInstr / 2; ++i) fetch_b(ys0a, 0, i);
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) fetch_a(xs1, BK, i);
#pragma unroll
    for (int i = kBInstr / 2; i < kBInstr; ++i) fetch_b(ys0b, 0, i);
#pragma unroll
    for (int i = 0; i < kBInstr / 2; ++i) fetch_b(ys1a, BK, i);
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) fetch_a(xs2, 2 * BK, i);
#pragma unroll
    for (int i = kBInstr / 2; i < kBInstr; ++i) fetch_b(ys1b, BK, i);
    __builtin_amdgcn_s_waitcnt(kWaitPrologue);  // x tile 0 and the first y half of tile 0 have landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) read_b(ys0a, b0, tn);
#pragma unroll
    for (int i = 0; i < TMH; ++i) read_a(xs0, 0, 0, af, i);

    // Tile kt lives in x_cur and the y halves (ya_cur, yb_cur); tile kt+1 in x_nxt, ya_nxt.
    auto k_tile = [&](unsigned char* x_cur, unsigned char* ya_cur, unsigned char* yb_cur, const unsigned char* x_nxt,
                      const unsigned char* ya_nxt, int kt) {
      // blocks: (K step 0, upper rows) (K step 0, lower rows) (K step 1, upper) (K step 1, lower); every block reads
      // the next block's x fragments, the second and the fourth also the next K step's y fragments
      block(af, b0, 0, x_cur, 0, 1, false, x_cur, b1, false, x_cur, x_cur, 0, 0, 0, 0);
      // First y half of tile kt is in registers everywhere; its second half has landed.
      __builtin_amdgcn_s_waitcnt(kWaitOlderLoads);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      block(af, b0, 1, x_cur, 1, 0, true, yb_cur, b1, false, x_cur, ya_cur, 0, kBInstr / 2, 0, (kt + 2) * BK);
      block(af, b1, 0, x_cur, 1, 1, false, x_cur, b0, false, x_cur, x_cur, 0, 0, 0, 0);
      // Hand-over: all of tile kt is in registers; x tile kt+1 and its first y half have landed.
      __builtin_amdgcn_s_waitcnt(kWaitOlderLoads);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      block(af, b1, 1, x_nxt, 0, 0, true, ya_nxt, b0, true, x_cur, yb_cur, kBInstr / 2, kBInstr, (kt + 3) * BK, (kt + 2) * BK);
    };
    // The stage names repeat every 6 tiles (3 x stages, 2 y stages).
    int kt = 0;
    for (; kt + 6 <= k_tiles; kt += 6) {
      k_tile(xs0, ys0a, ys0b, xs1, ys1a, kt);
      k_tile(xs1, ys1a, ys1b, xs2, ys0a, kt + 1);
      k_tile(xs2, ys0a, ys0b, xs0, ys1a, kt + 2);
      k_tile(xs0, ys1a, ys1b, xs1, ys0a, kt + 3);
      k_tile(xs1, ys0a, ys0b, xs2, ys1a, kt + 4);
      k_tile(xs2, ys1a, ys1b, xs0, ys0a, kt + 5);
    }
    const int rest = k_tiles - kt;
    if (rest > 0) k_tile(xs0, ys0a, ys0b, xs1, ys1a, kt);
    if (rest > 1) k_tile(xs1, ys1a, ys1b, xs2, ys0a, kt + 1);
    if (rest > 2) k_tile(xs2, ys0a, ys0b, xs0, ys1a, kt + 2);
    if (rest > 3) k_tile(xs0, ys1a, ys1b, xs1, ys0a, kt + 3);
    if (rest > 4) k_tile(xs1, ys0a, ys0b, xs2, ys1a, kt + 4);
    __builtin_amdgcn_s_waitcnt(0);  // trailing (zero-filling) fetches must not outlive the workgroup's LDS

    // Every wavefront is past its operand reads and every fetch has landed: the
    // stages are free to carry the output (two wavefronts share an x stage, the
    // last two take the y stages).
    __syncthreads();
    if (!combine(acc, reinterpret_cast<uint32_t*>(ys1b))) return;
    static_assert(2 * kEpilogueBytesPerWave<BAND> <= kABytes && kEpilogueBytesPerWave<BAND> <= kBBytes / 2 && kWaves <= 8,
                  "the output bands must fit the stages, and none lie in the last y half");
    unsigned char* band = wave < 2 ? xs0 : wave < 4 ? xs1 : wave < 6 ? xs2 : wave == 6 ? ys0a : ys0b;
    if (wave < 6) band += (wave & 1) * kEpilogueBytesPerWave<BAND>;
    store_tile_staged16<TM, TN, OutT, BAND>(acc, band, (OutT*)z.ptr, z.strides[0], z.shape[0], z.shape[1], row0 + wm * WM,
                                    col0 + wn * WN, lane, accumulate);
  }
};

}  // namespace gemm
}  // namespace cutile
