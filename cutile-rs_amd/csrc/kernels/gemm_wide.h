// GEMM tiles of 320 to 448 columns: one to a compute unit, most of the register file accumulators.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_common.h"
#include "kernel_args.h"

namespace cutile {
namespace gemm {

// BM x BN outputs on eight wavefronts (2 x 4, each BM / 2 rows by BN / 4 columns), K in tiles of 64, two LDS stages of x and two of y (y in halves of 32 K rows):
// one workgroup to a compute unit.  192 x 448 fills both memories: 160 KiB, and 168 accumulators of the 244 registers that a lane takes.
//
// What they are for: outputs whose last round of 256 x 256 or 192 x 256 tiles would leave most compute units idle, and which with the widths mixed
// (gemm_tiles.h) pay start and output of a tile twice; here they are one round, or two full ones.  A K tile of a full round costs 1.63, 1.78, 2.05 (192
// rows by 320, 384 and 448) and 1.99 us (256 x 320), 256 x 256 1.36 to 1.5: work by work the same rate, that of power and matrix issue, so they are the better ones only
// where they come out even.  f16, us before and here, operands from memory: 1500 x 14336 x 4096 165, 146 (192 x 448); 2048 x 8960 x 3584 133, 118; 1344 x
// 12032 x 4608 152, 124 (192 x 384); 560 x 28672 x 4096 142, 116; 1808 x 9344 x 10432 347, 288.  Same sums in the same order as on the other tiles of 64 K values.
//
// K step (32 wide) = TM / 2 pairs of row blocks; a pair is 2 TN MFMAs, column by column, so that a y fragment is free for the next K step's two MFMAs
// after the last pair has come to it, and is used again a whole pair later.  x fragments are two sets of a pair's two.
// Stages are refilled two K tiles ahead, as soon as every wavefront has read them: the first y half behind the barrier in K step 0, x and the
// second half behind the one in K step 1.  K is whole tiles: a fetch beyond the last one brings the last one again, which nobody reads.
// (256 x 384 has 192 accumulators, which leave too few registers: spills, 1500 x 14336 x 4096 197 us where the mix took 155.)
template <int BM_, int BN_, typename T>
struct GemmWide {
  static constexpr int BM = BM_, BN = BN_, BK = 64, kWaves = 8;
  static constexpr int WM = BM / 2, WN = BN / 4, TM = WM / 16, TN = WN / 16;
  static constexpr int PAIRS = TM / 2, SLOTS = 2 * TN;      // MFMAs of a pair
  static constexpr int UB = BN / 8, kPitch = BN * 2;        // 16-byte units and bytes of a y row
  static constexpr int kAInstr = BM / 64;                   // 1 KiB = 8 x rows; a wavefront's share
  // a y half is BN / 16 instructions; where that is no multiple of 8, four wavefronts take one more: the first four of the first half, the others of the second
  static constexpr int kBLeast = BN / 16 / kWaves, kBMost = (BN / 16 + kWaves - 1) / kWaves, kBTile = BN / 64;
  static constexpr int kABytes = BM * BK * 2, kBHalf = 32 * kPitch;
  static_assert(TM % 2 == 0 && BN % 64 == 0 && BM % 64 == 0, "row blocks in pairs; both halves together are the same share for every wavefront");

  struct Stages {
    unsigned char *xs0, *xs1, *ys0a, *ys0b, *ys1a, *ys1b;
  };

  // The accumulator stays in its registers: left to choose, the compiler gives the result others, and spills what it then lacks.  It does not know
  // this for a matrix instruction and puts no wait states behind it: nothing but MFMAs may touch the accumulators in the loop, so it must not spill there either.
  __device__ static __forceinline__ void mfma_in_place(const bf16x8& a, const bf16x8& b, f32x4& c) {
    if constexpr (__is_same(T, _Float16))
      asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
    else
      asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }

  __device__ static __forceinline__ int a_lds_off(int r, int u) { return r * (BK * 2) + ((u ^ ((r >> 1) & 7)) << 4); }
  // A transposing read takes 32 bytes of rows r .. r + 3 and r + 8 .. r + 11 at once, which are to lie in eight different eighths of 256 bytes: bits 0, 1 and 3 of
  // a row move it by 64, 128 and 32 bytes, bit 0 by itself where the pitch is an odd multiple of 128.
  static constexpr bool kOddPitch = kPitch % 256 != 0;
  __device__ static __forceinline__ int b_swizzle(int r) { return (kOddPitch ? ((r >> 1) & 1) << 2 : (r & 3) << 2) | (((r >> 3) & 1) << 1); }
  static constexpr int kSwizzled = kOddPitch ? 7 : 15;      // units among which the swizzle moves one

  __device__ static __forceinline__ void run_tile(const Stages& st, const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, int32_t k_total,
                                                  uint32_t pm, uint32_t pn, int32_t accumulate) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / 4, wn = wave % 4;
    const int32_t M = x.shape[0], N = y.shape[1], lda = x.strides[0], ldb = y.strides[0];
    const int32_t row0 = pm * BM, col0 = pn * BN;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(x.ptr, (uint32_t)(((int64_t)(M - 1) * lda + x.shape[1]) * 2));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(y.ptr, (uint32_t)(((int64_t)(y.shape[0] - 1) * ldb + N) * 2));
    constexpr uint32_t kOob = 0x80000000u;

    uint32_t a_goff[kAInstr], b_goff[kBMost];
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) {
      const int r = (wave * kAInstr + i) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
      a_goff[i] = row0 + r < M ? (uint32_t)(((int64_t)(row0 + r) * lda + u * 8) * 2) : kOob;
    }
    auto b_instr = [&](int i) { return i * kWaves + (i < kBLeast ? wave : wave & 3); };
#pragma unroll
    for (int i = 0; i < kBMost; ++i) {
      const int at = b_instr(i) * 64 + lane, r = at / UB, u = (at % UB) ^ b_swizzle(r);
      b_goff[i] = col0 + u * 8 < N ? (uint32_t)(((int64_t)r * ldb + col0 + u * 8) * 2) : kOob;
    }
    const int32_t k_tiles = k_total / BK, k_last = (k_tiles - 1) * BK;
    auto fetch_a = [&](unsigned char* stage, int32_t k0, int i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_PTR(void))(stage + (wave * kAInstr + i) * 1024), 16, a_goff[i], min(k0, k_last) * 2, 0, 0);
    };
    auto fetch_b = [&](unsigned char* half, int32_t k0, int h, int i) {
      if (i < kBLeast || (wave < 4) == (h == 0))
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LDS_PTR(void))(half + b_instr(i) * 1024), 16, b_goff[i], (min(k0, k_last) + 32 * h) * ldb * 2, 0, 0);
    };

    const int grp = lane >> 4, l16 = lane & 15, tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
    // One address each for x and y, from which the others are worked out where they are used: `fresh` keeps the compiler from holding all of them.
    int a_base = a_lds_off(wm * WM + l16, grp), b_base = (grp * 8 + tr_row) * kPitch + (((tr_col >> 3) ^ b_swizzle(grp * 8 + tr_row)) << 4) + (tr_col & 7) * 2;
    auto fresh = [](int& v) { asm volatile("" : "+v"(v)); };
    auto read_a = [&](const unsigned char* xs, int ks, int tm) { return *reinterpret_cast<const bf16x8*>(xs + (a_base ^ (ks << 6)) + tm * (16 * BK * 2)); };
    auto read_b = [&](const unsigned char* yh, int tn) {
      const int u = wn * (WN / 8) + tn * 2;   // unit of the fragment's first column; the swizzle moves a unit among 8 or 16
      const unsigned char* p = yh + (b_base ^ ((u & kSwizzled) << 4)) + ((u & ~kSwizzled) << 4);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 4 * kPitch));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    f32x4 acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0, 0, 0, 0};

    // Pair p of a K step on the x fragments `a`; reads the pair that comes next (row blocks 2 rd_p and 2 rd_p + 1 of K step rd_ks of rd_x) into `next`,
    // behind the last pair also the y fragments of the next K step from rd_y; deals out the refills of x_fill and y_fill.
    bf16x8 a0[2], a1[2], b[TN];
    auto pair = [&](bf16x8 (&a)[2], bf16x8 (&next)[2], int p, const unsigned char* rd_x, int rd_ks, int rd_p, bool last, const unsigned char* rd_y, bool with_x,
                    unsigned char* x_fill, bool with_y, unsigned char* y_fill, int half, int32_t k0) {
      fresh(a_base);
      if (last) fresh(b_base);
      const int n_fill = (with_x ? kAInstr : 0) + (with_y ? kBMost : 0);
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        const int tn = j / 2, h = j % 2;
        if (j < 2) next[j] = read_a(rd_x, rd_ks, 2 * rd_p + j);
#pragma unroll
        for (int i = 0; i < kAInstr + kBMost; ++i)
          if (i < n_fill && i * SLOTS / n_fill == j) {
            if (with_x && i < kAInstr)
              fetch_a(x_fill, k0, i);
            else
              fetch_b(y_fill, k0, half, i - (with_x ? kAInstr : 0));
          }
        mfma_in_place(b[tn], a[h], acc[tn][2 * p + h]);
        if (last && h == 1) b[tn] = read_b(rd_y, tn);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // s_waitcnt immediates: fetches that may still be in flight (vmcnt [3:0]); every LDS read done
    constexpr int kWaitHalf = (kBTile + kAInstr) | (7 << 4), kWaitTile = kBTile | (7 << 4), kWaitFirst = (kBLeast + kBTile + kAInstr) | (7 << 4);
    static_assert(kBLeast + kBTile + kAInstr <= 15, "the wait count must fit the low vmcnt field");

#pragma unroll
    for (int i = 0; i < kBMost; ++i) fetch_b(st.ys0a, 0, 0, i);
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) fetch_a(st.xs0, 0, i);
#pragma unroll
    for (int i = 0; i < kBMost; ++i) fetch_b(st.ys0b, 0, 1, i);
#pragma unroll
    for (int i = 0; i < kBMost; ++i) fetch_b(st.ys1a, BK, 0, i);
#pragma unroll
    for (int i = 0; i < kAInstr; ++i) fetch_a(st.xs1, BK, i);
#pragma unroll
    for (int i = 0; i < kBMost; ++i) fetch_b(st.ys1b, BK, 1, i);
    __builtin_amdgcn_s_waitcnt(kWaitFirst);   // x of tile 0 and its first y half
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) b[tn] = read_b(st.ys0a, tn);
    a0[0] = read_a(st.xs0, 0, 0), a0[1] = read_a(st.xs0, 0, 1);

    // (a K tile is an even number of pairs, and begins and ends on the same set of x fragments)
    auto k_tile = [&](unsigned char* x_cur, unsigned char* ya, unsigned char* yb, const unsigned char* x_nxt, const unsigned char* ya_nxt, int32_t kt) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          const bool last = p == PAIRS - 1, flip = (ks * PAIRS + p) % 2 != 0;
          if (last) {
            // K step 0: the second y half has landed; everyone has the first one in registers.  K step 1: x and the first y half of the next tile
            // have landed; everyone has this tile's x and second half in registers.
            if (ks == 0)
              __builtin_amdgcn_s_waitcnt(kWaitHalf);
            else
              __builtin_amdgcn_s_waitcnt(kWaitTile);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
          }
          const unsigned char* rx = last && ks == 1 ? x_nxt : x_cur;
          const int rks = last ? 1 - ks : ks, rp = last ? 0 : p + 1;
          pair(flip ? a1 : a0, flip ? a0 : a1, p, rx, rks, rp, last, ks == 0 ? yb : ya_nxt, last && ks == 1, x_cur, last, ks == 0 ? ya : yb, ks, (kt + 2) * BK);
        }
      }
    };
    for (int32_t kt = 0;;) {
      k_tile(st.xs0, st.ys0a, st.ys0b, st.xs1, st.ys1a, kt);
      if (++kt >= k_tiles) break;
      k_tile(st.xs1, st.ys1a, st.ys1b, st.xs0, st.ys0a, kt);
      if (++kt >= k_tiles) break;
    }
    __builtin_amdgcn_s_waitcnt(0);   // fetches beyond the last K tile must not outlive the workgroup's LDS
    __syncthreads();

    // The y stages carry the output, two bands to a half: 32 rows of a wavefront's sub-tile at a time (f32, chunk c of 16 bytes of row r at c ^ turn(r), which
    // with the pitch puts the 16 rows of one write on distinct banks); 16 lanes
    // then take a row, 8 columns each, and what lies outside z goes to an offset that the descriptor turns away.
    asm volatile("s_nop 15\n\ts_nop 15");   // the last MFMA's result, which the compiler does not know for one
    constexpr int kRow = WN * 4, kBand = 32 * kRow;
    static_assert(2 * kBand <= kBHalf, "the output bands must fit the stages");
    auto turn = [](int r) { return kRow % 128 == 0 ? (r >> 1) & 7 : (r >> 2) & 3; };
    static_assert(kRow % 256 == 128 || kRow % 128 == 64, "rows half of the banks apart, or a quarter");
    unsigned char* const ys = wave < 2 ? st.ys0a : wave < 4 ? st.ys0b : wave < 6 ? st.ys1a : st.ys1b;
    unsigned char* const band = ys + (wave & 1) * kBand;
    int e_lane = lane;
    fresh(e_lane);
    const int32_t zM = z.shape[0], zN = z.shape[1], ldz = z.strides[0];
    const __amdgpu_buffer_rsrc_t rz = make_rsrc(z.ptr, (uint32_t)(((int64_t)(zM - 1) * ldz + zN) * 2));
    const int rd_row = e_lane >> 4, rd_unit = e_lane & 15;
    const int32_t gc = col0 + wn * WN + rd_unit * 8;
    const bool col_ok = rd_unit < WN / 8 && gc < zN;
    const int unit = min(rd_unit, WN / 8 - 1);   // (the lanes of no column read what another one does)
    const bool stream = (int64_t)zM * zN * 2 >= kStreamedOutputBytes;
    auto offset = [&](int t, int pass) {
      const int32_t gr = row0 + wm * WM + t * 32 + pass * 4 + rd_row;
      return gr < zM && col_ok ? (uint32_t)(((int64_t)gr * ldz + gc) * 2) : kOob;
    };
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
      u32x4 old[8];
      if (accumulate) {
#pragma unroll
        for (int pass = 0; pass < 8; ++pass) old[pass] = __builtin_amdgcn_raw_buffer_load_b128(rz, offset(t, pass), 0, 0);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const int r = h * 16 + (e_lane & 15);
          *reinterpret_cast<f32x4*>(band + r * kRow + (((tn * 4 + (e_lane >> 4)) ^ turn(r)) << 4)) = acc[tn][2 * t + h];
        }
#pragma unroll
      for (int pass = 0; pass < 8; ++pass) {
        const int r = pass * 4 + rd_row;
        f32x4 lo = *reinterpret_cast<const f32x4*>(band + r * kRow + (((unit * 2) ^ turn(r)) << 4));
        f32x4 hi = *reinterpret_cast<const f32x4*>(band + r * kRow + (((unit * 2 + 1) ^ turn(r)) << 4));
        if (accumulate) {
          const u32x4 o = old[pass];
          lo[0] += stored_lo<T>(o.x), lo[1] += stored_hi<T>(o.x), lo[2] += stored_lo<T>(o.y), lo[3] += stored_hi<T>(o.y);
          hi[0] += stored_lo<T>(o.z), hi[1] += stored_hi<T>(o.z), hi[2] += stored_lo<T>(o.w), hi[3] += stored_hi<T>(o.w);
        }
        const u32x4 w = {pack_out2<T>(lo[0], lo[1]), pack_out2<T>(lo[2], lo[3]), pack_out2<T>(hi[0], hi[1]), pack_out2<T>(hi[2], hi[3])};
        if (stream)
          __builtin_amdgcn_raw_buffer_store_b128(w, rz, offset(t, pass), 0, 2);   // past the caches
        else
          __builtin_amdgcn_raw_buffer_store_b128(w, rz, offset(t, pass), 0, 0);
      }
    }
  }
};

}  // namespace gemm
}  // namespace cutile

// (the argument list of its family's members, gemm_tiles.h)
#define GEMM_WIDE_KERNEL(NAME, BM, BN, T)                                                                                                    \
  extern "C" __global__ void __launch_bounds__(512)                                                                                 \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k, TileGrid g, int32_t accumulate, float*,       \
                         uint32_t*, uint32_t) {                                                                                     \
    using Wide = GemmWide<BM, BN, T>;                                                                                                       \
    __shared__ __attribute__((aligned(1024))) unsigned char xs0[Wide::kABytes];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char xs1[Wide::kABytes];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char ys0a[Wide::kBHalf];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char ys0b[Wide::kBHalf];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char ys1a[Wide::kBHalf];                                                     \
    __shared__ __attribute__((aligned(1024))) unsigned char ys1b[Wide::kBHalf];                                                     \
    uint32_t pm, pn;                                                                                                                \
    tile_coords(g.x, g.y, &pm, &pn);                                                                                                \
    Wide::run_tile({xs0, xs1, ys0a, ys0b, ys1a, ys1b}, z, x, y, k, pm, pn, accumulate);                                             \
  }
