// MXFP8 GEMM on 128 x 128 tiles that have a compute unit to themselves (definition and operand layout: mxfp8_gemm.hip).
//
// Two stages of such a tile leave a fetch one K tile (0.2 us of matrix work) to land, less than one that misses L2 takes.  LDS holds four:
// tile kt + 3 goes into the stage that tile kt - 1 left, behind the one barrier at the start of tile kt.  By then every wavefront
// has multiplied with its last fragment of tile kt - 1 (a tile's fragments are read while the tile before it is multiplied, and are
// double-buffered), so nothing is waited for but the fetches of tile kt + 1, requested two K tiles ago.
// A row's 16 scale bytes serve four K tiles: they come with the first of these, go through one of two small buffers, and are read
// once into registers.  Every wavefront fetches its share of them twice over (64 rows a request, eight wavefronts, four shares), so
// that all wavefronts count the same requests.
// Neither pipe bounds it (counters, 200 x 14336 x 4096, of the clocks a compute unit is busy): the matrix pipes work 29 % of them, LDS 27 %, with no bank
// conflicts to speak of; a wavefront waits for fetches or at the barrier 37 % of them.  One workgroup of eight wavefronts to a compute unit has
// nobody to step in while all of it waits.
// Against the two stages (us): 200 x 14336 x 4096, 224 tiles, 24.8 -> 20.8; 1000 x 4096 x 4096, 256 tiles, 26.5 -> 22.3.
// The K tiles of an output tile may be shared by several workgroups, in whole scale blocks (split_k.h).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_common.h"
#include "kernel_args.h"
#include "split_k.h"

using namespace cutile;
using namespace cutile::gemm;

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));

template <typename OutT>
struct MxStages {
  static constexpr int BM = 128, BN = 128, BK = 128, WAVES_M = 2, WAVES_N = 4, kWaves = 8, kThreads = 512, STAGES = 4;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 16, TN = WN / 16, NB = TM * TN;
  static constexpr int kABytes = BM * BK, kStageBytes = (BM + BN) * BK, kScaleBytes = (BM + BN) * 16;
  static constexpr int kAInstr = BM / 8 / kWaves, kFetch = (BM + BN) / 8 / kWaves;   // 1 KiB = 8 rows of 128 bytes

  __device__ static __forceinline__ int lds_off(int r, int u) { return r * BK + ((u ^ ((r >> 1) & 7)) << 4); }
  static constexpr int wait_vm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }   // vmcnt(n) alone

  __device__ static __forceinline__ void run(const PartitionArg<2>& z, const TensorArg<2>& x, const TensorArg<2>& y, const TensorArg<2>& xs, const TensorArg<2>& ys,
                                             float alpha, const TileGrid& g, float* partials, uint32_t* counters, uint32_t splits) {
    __shared__ __attribute__((aligned(1024))) unsigned char st0[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st1[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st2[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st3[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char sc0[kScaleBytes];   // scale blocks 0, 2, 4 ...
    __shared__ __attribute__((aligned(1024))) unsigned char sc1[kScaleBytes];   // scale blocks 1, 3, 5 ...
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N, l16 = lane & 15, grp = lane >> 4;
    // split-major order: an XCD's contiguous share is neighbouring tiles on one range of K
    const uint32_t tiles_m = g.x, tiles_n = g.y, tiles = tiles_m * tiles_n, pos = xcd_contiguous(blockIdx.x, tiles * splits), split = pos / tiles, tile = pos % tiles;
    uint32_t pm, pn;
    grouped_tile(tile, tiles_m, tiles_n, &pm, &pn);
    const int32_t row0 = (int32_t)pm * BM, col0 = (int32_t)pn * BN;
    const int32_t M = x.shape[0], N = y.shape[0], K = min(x.shape[1], y.shape[1]);
    const int32_t all_tiles = K / BK, blocks = (all_tiles + 3) / 4;
    const int32_t first = (int32_t)((int64_t)blocks * split / splits) * 4, k_tiles = min((int32_t)((int64_t)blocks * (split + 1) / splits) * 4, all_tiles) - first;
    auto rsrc = [](const TensorArg<2>& t) { return make_rsrc(t.ptr, (uint32_t)((int64_t)(t.shape[0] - 1) * t.strides[0] + t.shape[1])); };
    const __amdgpu_buffer_rsrc_t ra = rsrc(x), rb = rsrc(y), rsa = rsrc(xs), rsb = rsrc(ys);
    constexpr uint32_t kOob = 0x80000000u;

    // Global side of the fetches (per lane, K tile `first`; the K advance is scalar).  Rows outside read zeros.
    uint32_t goff[kFetch];
#pragma unroll
    for (int i = 0; i < kFetch; ++i) {
      const bool is_x = i < kAInstr;
      const int r = (wave * kAInstr + (is_x ? i : i - kAInstr)) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
      goff[i] = is_x ? (row0 + r < M ? (uint32_t)((int64_t)(row0 + r) * x.strides[0] + u * 16) : kOob)
                     : (col0 + r < N ? (uint32_t)((int64_t)(col0 + r) * y.strides[0] + u * 16) : kOob);
    }
    const int share = wave & 3;   // of the scale rows: x 0..63, x 64..127, y 0..63, y 64..127
    const int s_row = (share & 1) * 64 + lane;
    const uint32_t s_goff = share < 2 ? (row0 + s_row < M ? (uint32_t)((int64_t)(row0 + s_row) * xs.strides[0]) : kOob)
                                      : (col0 + s_row < N ? (uint32_t)((int64_t)(col0 + s_row) * ys.strides[0]) : kOob);
    auto fetch = [&](unsigned char* stage, int32_t kt, int i) {
      const bool wanted = kt < k_tiles;   // past the last tile: zeros, which never leave the compute unit
      const int32_t k0 = wanted ? (first + kt) * BK : 0;
      const bool is_x = i < kAInstr;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(is_x ? ra : rb, (LDS_PTR(void))(stage + (is_x ? 0 : kABytes) + (wave * kAInstr + (is_x ? i : i - kAInstr)) * 1024), 16,
                                               wanted ? goff[i] : kOob, k0, 0, 0);
    };
    auto fetch_scales = [&](unsigned char* block, int32_t kt) {
      const bool wanted = kt < k_tiles;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(share < 2 ? rsa : rsb, (LDS_PTR(void))(block + share * 1024), 16, wanted ? s_goff : kOob, wanted ? (first + kt) * (BK / 32) : 0, 0, 0);
    };

    // LDS side: the lane's two 16-byte units of its row (K positions 16 g .. and 64 + 16 g ..); its scale is byte g of the tile's dword
    const int a_lo = lds_off(wm * WM + l16, grp), a_hi = lds_off(wm * WM + l16, 4 + grp);
    const int b_lo = kABytes + lds_off(wn * WN + l16, grp), b_hi = kABytes + lds_off(wn * WN + l16, 4 + grp);
    struct Frags {
      i32x8 a[TM], b[TN];
    };
    auto frag = [&](const unsigned char* lo, const unsigned char* hi) {
      const u32x4 l = *reinterpret_cast<const u32x4*>(lo), h = *reinterpret_cast<const u32x4*>(hi);
      return i32x8{(int)l.x, (int)l.y, (int)l.z, (int)l.w, (int)h.x, (int)h.y, (int)h.z, (int)h.w};
    };
    auto read = [&](const unsigned char* stage, Frags& f, int i) {
      if (i < TN)
        f.b[i] = frag(stage + b_lo + i * 16 * BK, stage + b_hi + i * 16 * BK);
      else
        f.a[i - TN] = frag(stage + a_lo + (i - TN) * 16 * BK, stage + a_hi + (i - TN) * 16 * BK);
    };
    u32x4 sa_blk[TM], sb_blk[TN];   // the scales of four K tiles
    auto read_scales = [&](const unsigned char* block) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) sa_blk[tm] = *reinterpret_cast<const u32x4*>(block + (wm * WM + tm * 16 + l16) * 16);
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) sb_blk[tn] = *reinterpret_cast<const u32x4*>(block + (BM + wn * WN + tn * 16 + l16) * 16);
    };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Tile kt (phase = kt % 4 = its stage) from fragments `f`; reads tile kt + 1 from `next`, fetches tile kt + 3 into `prev`.  `other`: the
    // buffer of the scale block after this tile's.
    auto k_tile = [&](const Frags& f, Frags& into, const unsigned char* next, unsigned char* prev, unsigned char* other, int32_t kt, auto phase) {
      constexpr int PH = decltype(phase)::value;
      // tile kt + 1 has landed: tile kt + 2 (with a scale block if it opens one) may be outstanding
      __builtin_amdgcn_s_waitcnt(wait_vm(kFetch + (PH == 2 ? 1 : 0)));
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t live = kt < k_tiles ? 0xffu : 0u;   // past the end lie another row's scales, which may be NaN
      int sa[TM], sb[TN];
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) sa[tm] = (int)((sa_blk[tm][PH] >> (8 * grp)) & live);
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) sb[tn] = (int)((sb_blk[tn][PH] >> (8 * grp)) & live);
      if constexpr (PH == 3) read_scales(other);
      constexpr int UNITS = TM + TN;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
#pragma unroll
        for (int i = 0; i < UNITS; ++i)
          if (i * (NB - 1) / UNITS == j) read(next, into, i);
#pragma unroll
        for (int i = 0; i < kFetch; ++i)
          if (i * NB / kFetch == j) fetch(prev, kt + 3, i);
        if (PH == 1 && j == NB - 1) fetch_scales(other, kt + 3);   // tile kt + 3 opens a scale block
        acc[j % TN][j / TN] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(f.b[j % TN], f.a[j / TN], acc[j % TN][j / TN], 0, 0, 0, sb[j % TN], 0, sa[j / TN]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    Frags f0, f1;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
      for (int i = 0; i < kFetch; ++i) fetch(t == 0 ? st0 : t == 1 ? st1 : st2, t, i);
      if (t == 0) fetch_scales(sc0, 0);
    }
    __builtin_amdgcn_s_waitcnt(wait_vm(2 * kFetch));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM + TN; ++i) read(st0, f0, i);
    read_scales(sc0);
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    using P2 = std::integral_constant<int, 2>;
    using P3 = std::integral_constant<int, 3>;
    int32_t kt = 0;
    auto four = [&](unsigned char* other) {
      k_tile(f0, f1, st1, st3, other, kt, P0{});
      k_tile(f1, f0, st2, st0, other, kt + 1, P1{});
      k_tile(f0, f1, st3, st1, other, kt + 2, P2{});
      k_tile(f1, f0, st0, st2, other, kt + 3, P3{});
      kt += 4;
    };
    while (kt < k_tiles) {   // whole scale blocks: tiles past the end are zeros times 2^-127
      four(sc1);
      if (kt >= k_tiles) break;
      four(sc0);
    }
    __builtin_amdgcn_s_waitcnt(0);   // trailing fetches must not outlive the workgroup's LDS
    __syncthreads();
    if (splits > 1 && !combine_tile<TM, TN, kThreads>(acc, partials + (size_t)tile * splits * (BM * BN), counters + tile, split, splits, reinterpret_cast<uint32_t*>(st3))) return;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) acc[tn][tm] *= alpha;
    static_assert(kWaves * kEpilogueBytesPerWave<WN> <= kStageBytes, "the output bands must fit a stage");
    store_tile_staged16<TM, TN, OutT>(acc, st0 + wave * kEpilogueBytesPerWave<WN>, (OutT*)z.ptr, z.strides[0], z.shape[0], z.shape[1], row0 + wm * WM, col0 + wn * WN, lane, 0);
  }
};

}  // namespace

#define MX_STAGES_KERNEL(NAME, OUT_T)                                                                                                \
  extern "C" __global__ void __launch_bounds__(512)                                                                                  \
      linear_tile_entry__##NAME(PartitionArg<2> z, TensorArg<2> x, TensorArg<2> y, TensorArg<2> xs, TensorArg<2> ys, float alpha,     \
                                TileGrid g, float* partials, uint32_t* counters, uint32_t splits) {                      \
    MxStages<OUT_T>::run(z, x, y, xs, ys, alpha, g, partials, counters, splits);                                                      \
  }
MX_STAGES_KERNEL(mxfp8_bf16_128x128x128_e2x2_lone, __bf16)
MX_STAGES_KERNEL(mxfp8_f32_128x128x128_e2x2_lone, float)
