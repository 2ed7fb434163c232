// GEMM bodies for the problems that leave the 256 x 256 macro-tiles of gemm_bf16.hip with too little to do: few rows of x
// (decoding, small batches).  Same tile program: z[M,N] (+)= x[M,K] . y[K,N], f32 accumulation, loads outside a tensor
// read 0, stores outside z are dropped.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_common.h"
#include "gemm_loose.h"
#include "gemm_thin.h"
#include "gemm_tiles.h"
#include "kernel_args.h"
#include "split_k.h"

using namespace cutile;
using namespace cutile::gemm;

namespace {

// ---- medium sizes: register-staged tiles, K split over workgroups -------------------------------------------------------
// For the outputs that are too few 256 x 256 tiles to fill the chip, and for rows that do not start on 16-byte boundaries
// (the direct global -> LDS fetches of gemm_bf16.hip cannot take those).  K tiles of 64 go global -> registers -> LDS: two
// tiles are in flight in registers while a third is multiplied out of one of two LDS stages.  The next tile is written to the other stage
// between the MFMAs of the first K step of 32, the one barrier lies between the two steps, and behind it the registers are loaded again: no
// phase of a K tile is without MFMAs, and the fragments of a step are read during the one before it.  Against phases of their own (multiply,
// write, load, barrier), us: f16 336 x 2575 x 1350 17.2 -> 14.6, 215 x 256 x 14720 21.8 -> 15.0, 1846 x 12923 x 374 50.9 -> 42.5; bf16 961 x 7277 x
// 2155 54.1 -> 44.0, 3136 x 1941 x 5340 99.6 -> 85.6.  With both operands unaligned a 128-byte piece of a row of x lies in two cache lines, which
// the vector cache does not hold until the next K tile: 2749 x 2583 x 8862 stays at 184.  Several workgroups may share the K tiles of a 64 x 64 output tile (SPLIT).
template <int BM, int BN, int WAVES_M, int WAVES_N, typename OutT, typename InT>
struct GemmStaged : StagedLayout<BN> {
  using Layout = StagedLayout<BN>;
  using Layout::a_lds_off, Layout::b_lds_off, Layout::load16;
  static constexpr bool SPLIT = BM == 64 && BN == 64;   // the tile that the launcher splits (staged_splits)
  static constexpr int BK = Layout::BK, UB = Layout::UB, kWaves = WAVES_M * WAVES_N, kThreads = kWaves * 64;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 16, TN = WN / 16;
  static constexpr int kALoads = BM * 8 / kThreads, kBLoads = BK * UB / kThreads;
  static constexpr int kABytes = BM * BK * 2, kBBytes = BK * BN * 2, kStageBytes = kABytes + kBBytes;
  static_assert(kALoads * kThreads == BM * 8 && kBLoads * kThreads == BK * UB && UB >= 8, "tile must split evenly");

  __device__ static void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, int32_t k_total, int32_t cover_m,
                             int32_t cover_n, int32_t accumulate, float* partials, uint32_t* counters, uint32_t tiles_m, uint32_t tiles_n,
                             uint32_t launch_splits) {
    const uint32_t splits = SPLIT ? launch_splits : 1;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kStageBytes];
    __shared__ uint32_t last;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N, l16 = lane & 15, grp = lane >> 4;
    // split-major order: an XCD's contiguous share is neighbouring tiles on one range of K
    const uint32_t tiles = tiles_m * tiles_n, pos = xcd_contiguous(blockIdx.x, tiles * splits), split = pos / tiles, tile = pos % tiles;
    const uint32_t per_group = kGroupM * tiles_n, first_m = tile / per_group * kGroupM, group_rows = min(tiles_m - first_m, (uint32_t)kGroupM);
    const uint32_t pm = first_m + tile % per_group % group_rows, pn = tile % per_group / group_rows;
    const int32_t M = x.shape[0], N = y.shape[1];
    const int64_t lda = (int64_t)x.strides[0] * 2, ldb = (int64_t)y.strides[0] * 2;   // bytes
    const int32_t k_valid = min(min(x.shape[1], y.shape[0]), k_total);
    const int32_t row0 = pm * BM, col_first = pn * BN, col0 = max(0, min(col_first, N - BN));   // the last column of tiles is moved back into y
    const int32_t k_tiles = (k_valid + BK - 1) / BK, kt0 = (int32_t)((int64_t)k_tiles * split / splits), kt1 = (int32_t)((int64_t)k_tiles * (split + 1) / splits);

    // per-lane byte offsets of the loads (operands end below 2 GiB; the K advance is scalar) and of the LDS writes
    static_assert(kThreads % 16 == 0 && kThreads / 8 % 16 == 0 && kThreads / UB % 16 == 0, "the swizzle terms repeat from load to load");
    const int a_r = tid / 8, b_r = tid / UB, a_k = tid % 8 * 8;
    uint32_t a_off[kALoads];
#pragma unroll
    for (int i = 0; i < kALoads; ++i)   // rows past the end repeat the last one and are not stored
      a_off[i] = (uint32_t)(min(row0 + a_r + i * (kThreads / 8), M - 1) * lda) + a_k * 2;
    const uint32_t b_off = (uint32_t)(b_r * ldb) + (uint32_t)(col0 + tid % UB * 8) * 2;
    const int64_t b_next = kThreads / UB * ldb;
    const int a_st = a_lds_off(a_r, tid % 8), b_st = kABytes + b_lds_off(b_r, tid % UB);
    const unsigned char* const xp = (const unsigned char*)x.ptr;
    const unsigned char* const yp = (const unsigned char*)y.ptr;
    struct Tile {
      u32x4 a[kALoads], b[kBLoads];
    };
    auto fetch_one = [&](Tile& t, int32_t kt, int i) {
      const int32_t k0 = kt * BK;
      if (i < kALoads)
        t.a[i] = load16(xp + (int64_t)k0 * 2 + a_off[i]);
      else
        t.b[i - kALoads] = load16(yp + k0 * ldb + (i - kALoads) * b_next + b_off);
    };
    // A ragged last K tile: K positions past the end are 0 on both sides.  Every unit of x is read where it lies inside K: one that the end cuts is
    // read so that it ends there, and shifted; y rows past the end repeat the last one, and give way to zeros (trim, when the tile is written).
    const int32_t rest = k_valid - (k_tiles - 1) * BK;
    const bool whole = a_k + 8 <= rest, partly = !whole && a_k < rest;
    auto ragged = [&](int32_t kt) { return __builtin_expect(kt == k_tiles - 1 && rest < BK, 0); };   // (out of the way of a short K)
    auto fetch_ragged = [&](Tile& t) {
      const int32_t k0 = (k_tiles - 1) * BK, at = whole ? k0 : k_valid - 8 - a_k;
#pragma unroll
      for (int i = 0; i < kALoads; ++i) {
        if (__builtin_expect(k_valid >= 8, 1)) {
          t.a[i] = load16(xp + a_off[i] + at * 2);
        } else {
          uint32_t o[4] = {0, 0, 0, 0};
          for (int e = 0; e < k_valid; ++e) {
            const uint32_t v = reinterpret_cast<const uint16_t*>(xp + a_off[i] - a_k * 2)[e];
#pragma unroll
            for (int d = 0; d < 4; ++d)
              if (e / 2 == d) o[d] |= v << (e % 2 * 16);
          }
          t.a[i] = u32x4{o[0], o[1], o[2], o[3]};
        }
      }
#pragma unroll
      for (int i = 0; i < kBLoads; ++i)
        t.b[i] = load16(yp + (int64_t)(k0 + min(b_r + i * (kThreads / UB), rest - 1)) * ldb + (b_off - (uint32_t)(b_r * ldb)));
    };
    auto trim = [&](Tile& t) {
      const int by = k_valid >= 8 ? (8 - rest % 8) % 8 * 16 : 0;   // bits that a cut unit was read too early, 16 to 112
#pragma unroll
      for (int i = 0; i < kALoads; ++i) {
        const uint64_t lo = t.a[i].x | (uint64_t)t.a[i].y << 32, hi = t.a[i].z | (uint64_t)t.a[i].w << 32;
        const uint64_t down = by == 0 ? lo : by < 64 ? lo >> by | hi << (64 - by) : hi >> (by - 64), up = by < 64 ? hi >> by : 0;
        const uint64_t nlo = whole ? lo : partly ? down : 0, nhi = whole ? hi : partly ? up : 0;
        t.a[i] = u32x4{(uint32_t)nlo, (uint32_t)(nlo >> 32), (uint32_t)nhi, (uint32_t)(nhi >> 32)};
      }
#pragma unroll
      for (int i = 0; i < kBLoads; ++i)
        if (b_r + i * (kThreads / UB) >= rest) t.b[i] = u32x4{0, 0, 0, 0};
    };
    auto fetch = [&](Tile& t, int32_t kt) {
      if (kt >= kt1) return;
      if (ragged(kt)) {
        fetch_ragged(t);
      } else {
#pragma unroll
        for (int i = 0; i < kALoads + kBLoads; ++i) fetch_one(t, kt, i);
      }
    };
    auto stage_one = [&](const Tile& t, unsigned char* s, int i) {
      if (i < kALoads)
        *reinterpret_cast<u32x4*>(s + a_st + i * (kThreads * 16)) = t.a[i];
      else
        *reinterpret_cast<u32x4*>(s + b_st + (i - kALoads) * (kThreads * 16)) = t.b[i - kALoads];
    };
    const int tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
    int a_addr[2], b_addr[TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_addr[ks] = a_lds_off(wm * WM + l16, ks * 4 + grp);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = wn * WN + tn * 16 + tr_col;
      b_addr[tn] = kABytes + b_lds_off(grp * 8 + tr_row, n >> 3) + (n & 7) * 2;   // rows r, r + 4, r + 32 share their swizzle term
    }
    f32x4 acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    struct Frags {
      bf16x8 a[TM], b[TN];
    };
    auto read = [&](const unsigned char* s, int ks, Frags& f, int i) {   // the y fragments and the first x fragment are needed first
      if (i < TN) {
        const unsigned char* p = s + b_addr[i] + ks * 32 * (BN * 2);
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
        s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 4 * (BN * 2)));
        f.b[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      } else {
        f.a[i - TN] = *reinterpret_cast<const bf16x8*>(s + a_addr[ks] + (i - TN) * (16 * BK * 2));
      }
    };
    // The MFMAs of a K step, and between them (sched_barrier keeps the order written) the reads of the next step's fragments, then what
    // moves the tiles along: writes of `t` to the stage `to`, or loads of K tile `load` into it.
    constexpr int NB = TM * TN, kUnits = TM + TN, kMoves = kALoads + kBLoads;
    constexpr std::integral_constant<int, 0> kNothing{};
    constexpr std::integral_constant<int, 1> kWrite{};
    constexpr std::integral_constant<int, 2> kLoad{};
    auto step = [&](const Frags& f, Frags& next, const unsigned char* rd, int rd_ks, bool reads, Tile& t, auto moves, unsigned char* to, int32_t load) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if (reads) {
#pragma unroll
          for (int i = 0; i < kUnits; ++i)
            if (i * NB / kUnits == j) read(rd, rd_ks, next, i);
        }
#pragma unroll
        for (int i = 0; i < kMoves; ++i)
          if (i * NB / kMoves == j) {
            if constexpr (decltype(moves)::value == 1) stage_one(t, to, i);
            if constexpr (decltype(moves)::value == 2) fetch_one(t, load, i);
          }
        acc[j % TN][j / TN] = mfma_16x16x32<InT>(f.b[j % TN], f.a[j / TN], acc[j % TN][j / TN]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    unsigned char* const s0 = lds;
    unsigned char* const s1 = lds + kStageBytes;
    Tile t0, t1;
    Frags f0, f1;
    if (kt0 < kt1) {
      fetch(t0, kt0);
      fetch(t1, kt0 + 1);
      if (ragged(kt0)) trim(t0);
#pragma unroll
      for (int i = 0; i < kMoves; ++i) stage_one(t0, s0, i);
      fetch(t0, kt0 + 2);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kUnits; ++i) read(s0, 0, f0, i);
    }
    // Tile kt lies in `cur`, tile kt + 1 in the registers `t` and, behind the barrier, in `next`: every wavefront has read its last fragment of
    // tile kt - 1 from there in front of the barrier of that tile.
    auto k_tile = [&](unsigned char* cur, unsigned char* next, Tile& t, int32_t kt, auto loads) {
      step(f0, f1, cur, 1, true, t, kWrite, next, 0);
      __syncthreads();
      step(f1, f0, next, 0, true, t, loads, next, kt + 3);
    };
    int32_t kt = kt0;
    for (; kt + 5 < kt1; kt += 2) {   // (the last K tile is not loaded in here)
      k_tile(s0, s1, t1, kt, kLoad);
      k_tile(s1, s0, t0, kt + 1, kLoad);
    }
#pragma unroll 1
    for (; kt < kt1; kt += 2) {       // (behind the last tile nothing is read that was written)
      if (ragged(kt + 1)) trim(t1);
      k_tile(s0, s1, t1, kt, kNothing);
      if (kt + 1 >= kt1) break;
      fetch(t1, kt + 3);
      if (ragged(kt + 2)) trim(t0);
      k_tile(s1, s0, t0, kt + 1, kNothing);
      fetch(t0, kt + 4);
    }

    const LooseOutput<OutT> out{(OutT*)z.ptr, z.strides[0], row0, col0, col_first, cover_m, cover_n, accumulate};
    const BlockPartials part(partials + (int64_t)tile * splits * (BM * BN), BM * BN * 4, splits);
    output_passes<BM, BN, WM, WN, kThreads, 2 * kStageBytes>(acc, lds, wm, wn, cover_m - row0, [&](int r, int u, f32x4 lo, f32x4 hi) {
      if (splits == 1) {
        const float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        out.template store<8>(r, u * 8, f);
      } else {
        part.store(split, (r * UB + u) * 2, lo);
        part.store(split, (r * UB + u) * 2 + 1, hi);
      }
    });
    if (splits == 1 || !last_to_arrive(counters + tile, splits, &last)) return;
    part.add_up<kThreads, 2>(min(BM, cover_m - row0) * (BN / 4), [&](int o, f32x4 v) {
      const float f[4] = {v[0], v[1], v[2], v[3]};
      out.template store<4>(o / (BN / 4), o % (BN / 4) * 4, f);
    });
  }
};

}  // namespace

#define GEMM_THIN_FAMILY(T, IN_T, OUT_T)               \
  GEMM_THIN_KERNEL(T##_thin16x64, IN_T, OUT_T, 1, 4, false)   \
  GEMM_THIN_KERNEL(T##_thin16x128, IN_T, OUT_T, 1, 8, false)  \
  GEMM_THIN_KERNEL(T##_thin32x64, IN_T, OUT_T, 2, 4, false)   \
  GEMM_THIN_KERNEL(T##_thin64x64, IN_T, OUT_T, 4, 4, false)
GEMM_THIN_FAMILY(bf16, __bf16, __bf16)
GEMM_THIN_FAMILY(f16, _Float16, _Float16)
GEMM_THIN_FAMILY(bf16f32, __bf16, float)

// (PER_SIMD wavefronts to a SIMD: as many workgroups on a compute unit as the launcher's prices say, host/gemm_choice.h)
#define GEMM_STAGED_KERNEL(NAME, IN_T, OUT_T, BM, BN, WVM, WVN, PER_SIMD)                                                           \
  extern "C" __global__ void __launch_bounds__(WVM * WVN * 64, PER_SIMD)                                                                   \
      gemm_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, int32_t k_total, int32_t cover_m, int32_t cover_n,       \
                         int32_t accumulate, float* partials, uint32_t* counters, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits) { \
    GemmStaged<BM, BN, WVM, WVN, OUT_T, IN_T>::run(z, x, y, k_total, cover_m, cover_n, accumulate, partials, counters, tiles_m,       \
                                                   tiles_n, splits);                                                                \
  }
#define GEMM_STAGED_FAMILY(T, IN_T, OUT_T)                     \
  GEMM_STAGED_KERNEL(T##_staged64x64, IN_T, OUT_T, 64, 64, 2, 2, 4)    \
  GEMM_STAGED_KERNEL(T##_staged64x128, IN_T, OUT_T, 64, 128, 2, 2, 3)  \
  GEMM_STAGED_KERNEL(T##_staged128x128, IN_T, OUT_T, 128, 128, 2, 2, 2) \
  GEMM_STAGED_KERNEL(T##_staged256x128, IN_T, OUT_T, 256, 128, 4, 2, 2)
GEMM_STAGED_FAMILY(bf16, __bf16, __bf16)
GEMM_STAGED_FAMILY(f16, _Float16, _Float16)
GEMM_STAGED_FAMILY(bf16f32, __bf16, float)

// ---- tiles between 128 x 128 and 256 x 256 (gemm_tiles.h) ----------------------------------------------------------------------
#define GEMM_TILES_FAMILY(N, T)                                  \
  GEMM_RING_TILE_KERNEL(N##_192x256x64_q2x4, 192, 256, 2, 4, T)       \
  GEMM_RING_TILE_KERNEL(N##_128x256x64_q2x4, 128, 256, 2, 4, T)       \
  GEMM_RING_TILE_KERNEL(N##_256x128x64_q4x2, 256, 128, 4, 2, T)       \
  GEMM_STAGES_KERNEL(N##_192x128x64_q2x2, 192, 128, 2, 4, 4, T)
GEMM_TILES_FAMILY(bf16, __bf16)
GEMM_TILES_FAMILY(f16, _Float16)
