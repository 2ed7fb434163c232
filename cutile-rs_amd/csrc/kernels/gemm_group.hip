// Grouped GEMM over descriptor tables on 128 x 128 tiles and on 256 x 256 ones (group_gemm_f16_nt_desc), for a launch of a workgroup to each compute unit:
// the reference's schedule (workgroup w computes tiles w, w + gridDim.x, ... of the groups' concatenated tiles), run ahead of itself.
//
// With few rows to a group the product is a read of the groups' B matrices, and what the ring kernel of that tile waited for was
// latency: it read the descriptors of one group after another until its tile's turn came (about 0.3 us each), started every tile with an
// empty pipeline, and had 1.25 K tiles of B in flight.  Here
//  * the descriptors of all groups are read at once, a thread to a group, into LDS with the groups' first tiles, and searched there;
//  * the operand stages run through from tile to tile: an iterator of its own walks the K tiles three ahead of the ones being
//    multiplied, across the ends of output tiles, and the output leaves from the accumulators, without LDS;
//  * B is read past the caches where no group has more than one row of tiles: then it is read once (16 groups of 96 x 6400 x 4608 on
//    average, some of two rows of tiles: 225 us through the caches, 241 past them).  us on the ring, here through the caches and here past them,
//    the same B again at once: 8 groups of 4096 x 2048 24.3, 24.2, 23.9; 32 of 1024 x 1024 24.2, 18.1, 17.2; 8 of 4096 x 4096, 268 MB, 45.4,
//    45.4, 45.3; sets of B in turn, so that it comes from memory: 27.8, 28.8, 25.8; 26.8, 18.7, 18.1; 49.1, 50.7, 46.4.  (B of 200 to 270 MB
//    that is just one tile to a compute unit is the one loss with B in the memory-side cache: 8 of 60 x 4096 x 3072 36.9, 37.2, 38.6);
//  * where the last round (the only one, or one behind others) has fewer tiles than half of the workgroups, several share the K tiles of one (split_k.h): 64 groups of
//    0 or 1 row x 1280 x 4352, 280 tiles, 78 -> 59 us; 16 of 2 or 3 x 3072 x 7168, 384, 129 -> 111; 16 of 92 x 3840 x 6400 214 -> 198.
// Stages, barriers and fragments as in GemmStages (gemm_tiles.h) with four stages.
// f16, us on the ring and here: 32 groups of 32 x 4096 x 4096 on average 200 and 183 (1.07 GB of B, 5.9 TB/s); 64 of 3.3 x 4608 x 7936
// 803 and 739; 64 of 2.4 x 768 x 512 36.8 and 19.2; sharing K, uneven groups, some without a row: 16 of 1 x 6912 x 1024 65.6 and 28.9 (52
// unshared), 8 of 8 x 6144 x 1792 60.7 and 35.5 (53).
#include <hip/hip_runtime.h>

#include "gemm_common.h"
#include "gemm_ring16.h"
#include "kernel_args.h"
#include "split_k.h"

using namespace cutile;
using namespace cutile::gemm;

namespace {

constexpr int kMostGroups = 256;   // the launcher sends no more (16 KiB of LDS)

struct Group {
  uint64_t a, b, c;                          // addresses
  int32_t m, k, n, lda, ldb, ldc, c_rows, c_cols;
  uint32_t first, tiles_n;                   // its first tile in the concatenated sequence, tiles to a tile row
};
static_assert(sizeof(Group) == 64, "");

struct GroupAhead {
  static constexpr int BM = 128, BN = 128, BK = 64, WAVES_N = 2, kWaves = 8, kThreads = 512, STAGES = 4;
  static constexpr int WM = 32, WN = 64, TM = 2, TN = 4, NB = TM * TN, UB = BN / 8;
  static constexpr int kAInstr = 2, kBRows = 64 / UB, kBInstr = 2, kFetch = kAInstr + kBInstr;
  static constexpr int kABytes = BM * BK * 2, kStageBytes = kABytes + BK * BN * 2;
  static constexpr int kNontemporal = 2;
  static constexpr uint32_t kOob = 0x80000000u;   // out of range of every resource made here
  // K tiles that a sharing workgroup gets at least: the sum costs 3 to 4 us, a K tile 0.4 (16 groups of 1 x 1280 x 512 in threes 14.1 ->
  // 12.6 us; 8 of 11 x 768 x 2048, 12 K tiles in twos, 11.9 -> 13.4)
  static constexpr uint32_t kFewestPerSplit = 8;

  __device__ static __forceinline__ int a_lds_off(int r, int u) { return r * (BK * 2) + ((u ^ ((r >> 1) & 7)) << 4); }
  __device__ static __forceinline__ int b_swizzle(int r) { return ((r & 3) << 2) | (((r >> 3) & 1) << 1); }
  __device__ static __forceinline__ int b_lds_off(int r, int u) { return r * (BN * 2) + ((u ^ b_swizzle(r)) << 4); }
  static constexpr int wait_vm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }   // vmcnt(n) alone
  __device__ static __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
  __device__ static __forceinline__ uint64_t uniform64(uint64_t v) {
    return (uint64_t)(uint32_t)uniform((int32_t)(uint32_t)v) | (uint64_t)(uint32_t)uniform((int32_t)(uint32_t)(v >> 32)) << 32;
  }

  struct Stage {
    unsigned char *a, *b;
  };
  // What the workgroup knows of the launch before it starts: a thread to a group its descriptors, and how many tiles of 128 x 128 and of 256 x 256 lie in front of it.
  struct Survey {
    Group d;
    uint32_t before, before_wide, total, total_wide, most_k, most_m;
  };
  template <bool WIDE>
  __device__ static __forceinline__ Survey survey(const TensorArg<1>& a_ptrs, const TensorArg<1>& b_ptrs, const TensorArg<1>& c_ptrs, const TensorArg<2>& a_metas,
                                                  const TensorArg<2>& b_metas, const TensorArg<2>& c_metas, int32_t num_groups, uint32_t* scratch) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t *const wave_tiles = scratch, *const wave_k = scratch + 4, *const wave_m = scratch + 8, *const wave_wide = scratch + 12;
    Survey v{};
    uint32_t mine = 0, wide = 0;
    if (tid < num_groups) {
      Group& d = v.d;
      auto address = [&](const TensorArg<1>& t) { return (uint64_t)((const int64_t*)t.ptr)[(int64_t)tid * t.strides[0]]; };
      auto meta = [&](const TensorArg<2>& t, int i) { return ((const int32_t*)t.ptr)[(int64_t)tid * t.strides[0] + i * t.strides[1]]; };
      d.a = address(a_ptrs), d.b = address(b_ptrs), d.c = address(c_ptrs);
      d.m = meta(a_metas, 0), d.k = min(meta(a_metas, 1), meta(b_metas, 0)), d.lda = meta(a_metas, 2);
      d.n = meta(b_metas, 1), d.ldb = meta(b_metas, 2);
      d.c_rows = meta(c_metas, 0), d.c_cols = meta(c_metas, 1), d.ldc = meta(c_metas, 2);
      d.tiles_n = (uint32_t)((d.n + BN - 1) / BN);
      mine = (uint32_t)((d.m + BM - 1) / BM) * d.tiles_n;
      if constexpr (WIDE) wide = (uint32_t)((d.m + 2 * BM - 1) / (2 * BM)) * (uint32_t)((d.n + 2 * BN - 1) / (2 * BN));
    }
    // running sums and maxima over the first four wavefronts, in as many steps as there are groups for
    uint32_t sum = mine, sum_wide = wide, most_k = mine ? (uint32_t)((v.d.k + BK - 1) / BK) : 0, most_m = mine ? (uint32_t)v.d.m : 0;
    for (int o = 1; o < min(num_groups, 64); o <<= 1) {
      const uint32_t below = __shfl_up(sum, o, 64), below_wide = WIDE ? __shfl_up(sum_wide, o, 64) : 0;
      if (lane >= o) sum += below, sum_wide += below_wide;
      most_k = max(most_k, (uint32_t)__shfl_xor(most_k, o, 64)), most_m = max(most_m, (uint32_t)__shfl_xor(most_m, o, 64));
    }
    if (lane == min(num_groups - 1, 63) && wave < 4) wave_tiles[wave] = sum, wave_k[wave] = most_k, wave_m[wave] = most_m, wave_wide[wave] = sum_wide;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave && wave < 4) sum += wave_tiles[w], sum_wide += wave_wide[w];
      v.total += wave_tiles[w], v.total_wide += wave_wide[w];
      v.most_k = max(v.most_k, wave_k[w]), v.most_m = max(v.most_m, wave_m[w]);
    }
    v.total = (uint32_t)uniform((int32_t)v.total), v.total_wide = (uint32_t)uniform((int32_t)v.total_wide);
    v.most_k = (uint32_t)uniform((int32_t)v.most_k), v.most_m = (uint32_t)uniform((int32_t)v.most_m);
    v.before = sum - mine, v.before_wide = sum_wide - wide;
    return v;
  }

  __device__ static __forceinline__ void run(const TensorArg<1>& a_ptrs, const TensorArg<1>& b_ptrs, const TensorArg<1>& c_ptrs, const TensorArg<2>& a_metas,
                                             const TensorArg<2>& b_metas, const TensorArg<2>& c_metas, int32_t num_groups, float* partials, uint32_t* counters) {
    __shared__ __attribute__((aligned(1024))) unsigned char st0[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st1[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st2[kStageBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char st3[kStageBytes];
    __shared__ __attribute__((aligned(16))) Group groups[kMostGroups];
    __shared__ uint32_t scratch[16];
    if (num_groups == 0) return;
    Survey v = survey<false>(a_ptrs, b_ptrs, c_ptrs, a_metas, b_metas, c_metas, num_groups, scratch);
    if ((int)threadIdx.x < num_groups) {
      v.d.first = v.before;
      groups[threadIdx.x] = v.d;
    }
    __syncthreads();
    run_tiles(groups, num_groups, v.total, shares_of(v.total, v.most_k, partials), v.most_m, partials, counters, Stage{st0, st0 + kABytes}, Stage{st1, st1 + kABytes},
              Stage{st2, st2 + kABytes}, Stage{st3, st3 + kABytes}, scratch);
  }

  // How many workgroups share the K of each tile of the last round, where that has fewer tiles than half of the workgroups.
  __device__ static __forceinline__ uint32_t shares_of(uint32_t total, uint32_t most_k, const float* partials) {
    const uint32_t grid = gridDim.x, rest = total < grid ? total : total % grid;
    return partials && rest && 2 * rest <= grid ? max(1u, min(grid / rest, most_k / kFewestPerSplit)) : 1u;
  }
  __device__ static __forceinline__ void run_tiles(const Group* groups, int32_t num_groups, uint32_t total, uint32_t splits, uint32_t most_m, float* partials, uint32_t* counters,
                                                   Stage st0, Stage st1, Stage st2, Stage st3, uint32_t* flag) {
    const bool once = most_m <= BM;
    if (splits > 1) {
      const uint32_t whole = total < gridDim.x ? 0 : total / gridDim.x * gridDim.x;
      if (blockIdx.x >= (total - whole) * splits && whole == 0) return;
      once ? walk<true, true>(groups, num_groups, total, whole, splits, partials, counters, st0, st1, st2, st3, flag)
           : walk<false, true>(groups, num_groups, total, whole, splits, partials, counters, st0, st1, st2, st3, flag);
    } else if (blockIdx.x < total) {
      once ? walk<true, false>(groups, num_groups, total, total, 1, partials, counters, st0, st1, st2, st3, flag)
           : walk<false, false>(groups, num_groups, total, total, 1, partials, counters, st0, st1, st2, st3, flag);
    }
  }

  // ONCE: no group has more than one row of tiles.  SHARE: the tiles before `whole` are dealt out one to a workgroup and round, those behind it to `splits` workgroups each.
  template <bool ONCE, bool SHARE>
  __device__ static __forceinline__ void walk(const Group* groups, int32_t num_groups, uint32_t total, uint32_t whole, uint32_t splits, float* partials, uint32_t* counters,
                                              Stage st0, Stage st1, Stage st2, Stage st3, uint32_t* flag) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const uint32_t rest = total - whole, split = SHARE ? blockIdx.x / rest : 0;
    const uint32_t shared_tile = SHARE && split < splits ? whole + blockIdx.x - split * rest : total;   // total: none
    // The tiles of this workgroup, one after another (two such walks: of the tiles being fetched and of the one being multiplied).
    struct Walk {
      uint32_t tile;
      int32_t group;
    };
    auto next_tile = [&](uint32_t tile) {   // at or past `total`: no more
      const uint32_t on = tile + gridDim.x;
      return !SHARE || on < whole ? on : tile < whole ? shared_tile : total;
    };
    auto find = [&](Walk& w) {   // the last group that begins at or before the tile and has tiles
      while (w.group + 1 < num_groups && (uint32_t)uniform((int32_t)groups[w.group + 1].first) <= w.tile) ++w.group;
    };
    // K tiles [k0, k1) of this workgroup, at least one (of zeros, where there are none)
    auto k_range = [&](uint32_t tile, int32_t k, int32_t* k0, int32_t* k1) {
      const int32_t n = (k + BK - 1) / BK;
      *k0 = 0, *k1 = n;
      if (!SHARE || tile < whole) return;
      const int32_t each = n / (int32_t)splits, more = n % (int32_t)splits;
      *k0 = each * (int32_t)split + min((int32_t)split, more), *k1 = *k0 + each + ((int32_t)split < more);
    };
    auto k_tiles_of = [&](const Walk& w) {
      int32_t k0, k1;
      k_range(w.tile, uniform(groups[w.group].k), &k0, &k1);
      return max(1, k1 - k0);
    };

    // ---- fetching ----
    Walk fw{SHARE && blockIdx.x >= whole ? shared_tile : blockIdx.x, 0};
    __amdgpu_buffer_rsrc_t ra, rb;
    uint32_t a_goff[kAInstr], b_goff[kBInstr];
    int32_t f_k = 0, f_kt = 0, f_tiles = 0, f_ldb = 0;
    auto fetch_tile_of = [&] {   // points the fetches at tile fw.tile, or out of range past the last one
      const bool live = fw.tile < total;
      if (live) find(fw);
      const Group& g = groups[fw.group];
      const int32_t m = uniform(g.m), n = uniform(g.n), lda = uniform(g.lda), k = uniform(g.k), ldb = uniform(g.ldb);
      const uint32_t in_group = fw.tile - (uint32_t)uniform((int32_t)g.first), tiles_n = (uint32_t)max(1, uniform((int32_t)g.tiles_n));
      const int32_t row0 = (int32_t)(in_group / tiles_n) * BM, col0 = (int32_t)(in_group % tiles_n) * BN;
      int32_t k0, k1;
      k_range(fw.tile, k, &k0, &k1);
      f_k = live ? min(k, k1 * BK) : 0, f_kt = live ? k0 : 0, f_tiles = live ? max(k0 + 1, k1) : 0x7fffffff, f_ldb = ldb;
      // (past the last tile the position in the group means nothing: no byte is in range)
      const bool any = live && k > 0;
      ra = make_rsrc((const uint16_t*)uniform64(g.a) + (any ? (int64_t)row0 * lda : 0), any ? (uint32_t)(((int64_t)(min(m - row0, BM) - 1) * lda + k) * 2) : 0u);
      rb = make_rsrc((const void*)uniform64(g.b), any ? (uint32_t)(((int64_t)(k - 1) * ldb + n) * 2) : 0u);
#pragma unroll
      for (int i = 0; i < kAInstr; ++i) {
        const int r = (wave * kAInstr + i) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
        a_goff[i] = row0 + r < m ? (uint32_t)((r * lda + u * 8) * 2) : kOob;
      }
#pragma unroll
      for (int i = 0; i < kBInstr; ++i) {
        const int r = (i * kWaves + wave) * kBRows + lane / UB, u = (lane % UB) ^ b_swizzle(r);
        b_goff[i] = col0 + u * 8 < n ? (uint32_t)(((int64_t)r * ldb + col0 + u * 8) * 2) : kOob;
      }
    };
    // request i of the K tile that the fetches have come to (K positions past the end bring zeros: K is a multiple of 8)
    auto fetch = [&](const Stage& stage, int i) {
      const int32_t k0 = f_kt * BK;
      if (i < kAInstr) {
        const int r = (wave * kAInstr + i) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_PTR(void))(stage.a + (wave * kAInstr + i) * 1024), 16, k0 + u * 8 < f_k ? a_goff[i] : kOob,
                                                 k0 < f_k ? k0 * 2 : 0, 0, 0);
      } else {
        const int b = i - kAInstr, r = (b * kWaves + wave) * kBRows;
        const LDS_PTR(void) to = (LDS_PTR(void))(stage.b + (b * kWaves + wave) * 1024);
        const uint32_t off = k0 + r + (lane / UB) < f_k ? b_goff[b] : kOob;
        const int32_t at = k0 < f_k ? k0 * f_ldb * 2 : 0;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, to, 16, off, at, 0, ONCE ? kNontemporal : 0);
      }
    };
    auto fetched = [&] {   // on to the next K tile
      if (++f_kt == f_tiles) {
        fw.tile = next_tile(fw.tile);
        fetch_tile_of();
      }
    };

    // ---- multiplying ----
    const int grp = lane >> 4, l16 = lane & 15, tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
    int a_addr[2], b_addr[TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_addr[ks] = a_lds_off(wm * WM + l16, ks * 4 + grp);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = wn * WN + tn * 16 + tr_col;
      b_addr[tn] = b_lds_off(grp * 8 + tr_row, n >> 3) + (n & 7) * 2;
    }
    struct Frags {
      bf16x8 a[TM], b[TN];
    };
    auto read = [&](const Stage& stage, int ks, Frags& f, int i) {
      if (i < TN) {
        const unsigned char* p = stage.b + b_addr[i] + ks * 32 * (BN * 2);
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
        s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 4 * (BN * 2)));
        f.b[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      } else {
        f.a[i - TN] = *reinterpret_cast<const bf16x8*>(stage.a + a_addr[ks] + (i - TN) * (16 * BK * 2));
      }
    };
    f32x4 acc[TN][TM];
    auto clear = [&] {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    constexpr int UNITS = TM + TN;
    auto step = [&](const Frags& f, Frags& next, const Stage& rd, int rd_ks, bool fill, const Stage& fill_stage) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
#pragma unroll
        for (int i = 0; i < UNITS; ++i)
          if (i * (NB - 1) / UNITS == j) read(rd, rd_ks, next, i);
        if (fill) {
#pragma unroll
          for (int i = 0; i < kFetch; ++i)
            if (i * NB / kFetch == j) fetch(fill_stage, i);
        }
        acc[j % TN][j / TN] = mfma_16x16x32<_Float16>(f.b[j % TN], f.a[j / TN], acc[j % TN][j / TN]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    Walk cw = fw;
    int32_t c_left = 0;   // K tiles that the tile being multiplied still has
    find(cw);
    c_left = k_tiles_of(cw);
    clear();
    // lane (grp, l16) holds row l16 of each 16-row block and columns 4 grp .. + 3 of each 16-column block
    auto store = [&] {
      const Group& g = groups[cw.group];
      const int32_t rows = uniform(g.c_rows), cols = uniform(g.c_cols), ldc = uniform(g.ldc);
      const uint32_t in_group = cw.tile - (uint32_t)uniform((int32_t)g.first), tiles_n = (uint32_t)uniform((int32_t)g.tiles_n);
      const int32_t row0 = (int32_t)(in_group / tiles_n) * BM, col0 = (int32_t)(in_group % tiles_n) * BN;
      uint16_t* const c = (uint16_t*)uniform64(g.c) + (int64_t)row0 * ldc + col0;
      const int32_t left_m = min(rows - row0, BM), left_n = min(cols - col0, BN), r0 = wm * WM + l16, c0 = wn * WN + grp * 4;
      const __amdgpu_buffer_rsrc_t rc = make_rsrc(c, left_m > 0 && left_n > 0 ? (uint32_t)(((int64_t)(left_m - 1) * ldc + left_n) * 2) : 0u);
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const int r = r0 + tm * 16, col = c0 + tn * 16;
          const uint32_t off = (uint32_t)((r * ldc + col) * 2);
          const u32x2 v = {pack_out2<_Float16>(acc[tn][tm][0], acc[tn][tm][1]), pack_out2<_Float16>(acc[tn][tm][2], acc[tn][tm][3])};
          __builtin_amdgcn_raw_buffer_store_b64(v, rc, r < left_m && col < left_n ? off : kOob, 0, 0);
        }
    };
    Frags f0, f1;
    // one K tile from stage `cur`: its second half's fragments, then, behind the barrier, the next tile's first ones and the fetch of the third tile on
    auto k_tile = [&](const Stage& cur, const Stage& next, const Stage& prev) {
      step(f0, f1, cur, 1, false, prev);
      __builtin_amdgcn_s_waitcnt(wait_vm((STAGES - 3) * kFetch));
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      step(f1, f0, next, 0, true, prev);
      fetched();
      if (--c_left == 0 && (!SHARE || cw.tile < whole)) {   // (past the last tile, and of a shared one, it goes on below 0)
        store();
        clear();
        cw.tile = next_tile(cw.tile);
        if (cw.tile < total) {
          find(cw);
          c_left = k_tiles_of(cw);
        }
      }
    };
    fetch_tile_of();
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) {
#pragma unroll
      for (int i = 0; i < kFetch; ++i) fetch(s == 0 ? st0 : s == 1 ? st1 : st2, i);
      fetched();
    }
    __builtin_amdgcn_s_waitcnt(wait_vm((STAGES - 2) * kFetch));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < UNITS; ++i) read(st0, 0, f0, i);
    do {   // (up to three K tiles of zeros at the end: leaving from each of the four places would cost the loop a full wait)
      k_tile(st0, st1, st3);
      k_tile(st1, st2, st0);
      k_tile(st2, st3, st1);
      k_tile(st3, st0, st2);
    } while (SHARE ? cw.tile < whole || (cw.tile < total && c_left > 0) : cw.tile < total);
    __builtin_amdgcn_s_waitcnt(0);   // trailing (zero-filling) fetches must not outlive the workgroup's LDS
    if (SHARE && cw.tile < total) {   // a shared one
      constexpr uint32_t kTile = BM * BN * 4;
      const Group& g = groups[cw.group];
      const uint32_t in_group = cw.tile - (uint32_t)uniform((int32_t)g.first), tiles_n = (uint32_t)uniform((int32_t)g.tiles_n);
      const bool active = (int32_t)(in_group / tiles_n) * BM + wm * WM < uniform(g.c_rows);   // (wavefronts without a row to store hold nothing)
      const __amdgpu_buffer_rsrc_t part = make_rsrc(partials + (size_t)(cw.tile - whole) * splits * (BM * BN), kTile * splits);
      if (active) {
#pragma unroll
        for (int r = 0; r < NB; ++r) store_partial(acc[r % TN][r / TN], part, split * kTile + r * (kThreads * 16) + threadIdx.x * 16);
      }
      if (!last_to_arrive(counters + (cw.tile - whole), splits, flag) || !active) return;
      clear();
      for (uint32_t k = 0; k < splits; ++k)
#pragma unroll
        for (int r = 0; r < NB; ++r)
          acc[r % TN][r / TN] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(part, threadIdx.x * 16, k * kTile + r * (kThreads * 16), kAgentScope));
      store();
    }
  }
};

// Launches of 256 x 256 tiles: on those (the ring of gemm_ring16.h, tile after tile), or on the 128 x 128 ones above where that is sooner done.  Which of the two only the
// descriptors say, so the workgroups decide, all alike.  What the ring alone waited for were descriptors, read group after group (0.3 us each, 64 groups of 135 x 2048 x 1792 153 -> 125 us, now
// read at once), and rounds that left most compute units idle or had a handful of tiles (16 groups of 252 x 512 x 1280, 46 tiles of 256 x 256, 40 -> 20 us; 8 of 251 x 5632 x 6656,
// 264 tiles, 312 -> 268).  60 drawn launches 0.89 of their time, from 0.52 to 1.03 (8 and 16 groups that have nothing to gain: about a microsecond for the sums over the groups).
struct GroupWide {
  using Ring = GemmRing16<256, 256, 2, 4, _Float16, _Float16>;
  using Ahead = GroupAhead;
  static_assert(Ring::kABytes == Ahead::kStageBytes && Ring::kBBytes / 2 == Ahead::kABytes && sizeof(Group) * kMostGroups <= Ring::kBBytes / 2, "one set of LDS arrays serves both");

  __device__ static __forceinline__ void run(const TensorArg<1>& a_ptrs, const TensorArg<1>& b_ptrs, const TensorArg<1>& c_ptrs, const TensorArg<2>& a_metas,
                                             const TensorArg<2>& b_metas, const TensorArg<2>& c_metas, int32_t num_groups, float* partials, uint32_t* counters) {
    __shared__ __attribute__((aligned(1024))) unsigned char xs0[Ring::kABytes];
    __shared__ __attribute__((aligned(1024))) unsigned char xs1[Ring::kABytes];
    __shared__ __attribute__((aligned(1024))) unsigned char xs2[Ring::kABytes];
    __shared__ __attribute__((aligned(1024))) unsigned char ys0a[Ring::kBBytes / 2];
    __shared__ __attribute__((aligned(1024))) unsigned char ys0b[Ring::kBBytes / 2];
    __shared__ __attribute__((aligned(1024))) unsigned char ys1a[Ring::kBBytes / 2];
    __shared__ __attribute__((aligned(1024))) unsigned char ys1b[Ring::kBBytes / 2];
    if (num_groups == 0) return;
    uint32_t* const scratch = reinterpret_cast<uint32_t*>(ys1b);
    Group* const groups = reinterpret_cast<Group*>(ys1a);
    Ahead::Survey v = Ahead::survey<true>(a_ptrs, b_ptrs, c_ptrs, a_metas, b_metas, c_metas, num_groups, scratch);
    const uint32_t grid = gridDim.x, splits = Ahead::shares_of(v.total, v.most_k, partials);
    // us, fitted to 60 drawn launches of 8 to 64 groups (K 512 to 6700, 16 to 2400 tiles of 256 x 256): the pick takes 1.002 of the better one's time
    const uint32_t full = v.total / grid, rest = v.total - full * grid, wide_rounds = (v.total_wide + grid - 1) / grid;
    const float k = (float)v.most_k, rounds = (float)full + (rest ? __builtin_amdgcn_rcpf((float)splits) : 0.0f);
    const float narrow = 12.7f + rounds * k * 0.705f + (float)(full + (rest ? 1 : 0)) * 1.7f + (splits > 1 ? 4.9f : 0.0f), wide = (float)wide_rounds * (k * 1.55f + 13.7f);
    const bool take_narrow = narrow < 0.85f * wide;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < num_groups) {
      v.d.first = take_narrow ? v.before : v.before_wide;
      groups[tid] = v.d;
    }
    __syncthreads();
    if (take_narrow) {
      Ahead::run_tiles(groups, num_groups, v.total, splits, v.most_m, partials, counters, Ahead::Stage{xs0, xs0 + Ahead::kABytes}, Ahead::Stage{xs1, xs1 + Ahead::kABytes},
                       Ahead::Stage{xs2, xs2 + Ahead::kABytes}, Ahead::Stage{ys0a, ys0b}, scratch);
      return;
    }
    // Lane r finds the group of the workgroup's r-th tile, as the table's LDS belongs to the stages from here on; the first kFound are kept, in scalar registers (beside the
    // ring's there is no vector register to spare).
    constexpr int kFound = 4;
    int32_t found_group[kFound], found_place[kFound];
    {
      const uint32_t tile = blockIdx.x + lane * grid;
      int32_t lo = 0, hi = num_groups;   // the last group that begins at or before the tile is in [lo, hi)
      while (hi - lo > 1) {
        const int32_t mid = (lo + hi) >> 1;
        (groups[mid].first <= tile ? lo : hi) = mid;
      }
      const int32_t place = (int32_t)(tile - groups[lo].first);
#pragma unroll
      for (int i = 0; i < kFound; ++i) found_group[i] = __builtin_amdgcn_readlane(lo, i), found_place[i] = __builtin_amdgcn_readlane(place, i);
    }
    __syncthreads();
    auto uniform = [](int32_t x) { return __builtin_amdgcn_readfirstlane(x); };
    auto describe = [&](const TensorArg<1>& ptrs, const TensorArg<2>& metas, int32_t g, TensorArg<2>* t) {
      const uint32_t* pp = reinterpret_cast<const uint32_t*>((const int64_t*)ptrs.ptr + (int64_t)g * ptrs.strides[0]);
      const int32_t* mp = (const int32_t*)metas.ptr + (int64_t)g * metas.strides[0];
      t->ptr = (void*)((uint64_t)(uint32_t)uniform((int32_t)pp[0]) | ((uint64_t)(uint32_t)uniform((int32_t)pp[1]) << 32));
      t->shape[0] = uniform(mp[0]);
      t->shape[1] = uniform(mp[metas.strides[1]]);
      t->strides[0] = uniform(mp[2 * metas.strides[1]]);
      t->strides[1] = 1;
    };
    int32_t group = 0;
    uint32_t place = 0, r = 0;
    for (uint32_t tile = blockIdx.x; tile < v.total_wide; tile += grid, ++r) {
      place += grid;   // in the group of the tile before, or behind it
#pragma unroll
      for (int i = 0; i < kFound; ++i)
        if (r == (uint32_t)i) group = found_group[i], place = (uint32_t)found_place[i];
      TensorArg<2> a, b, c;
      uint32_t tiles_n;
      for (;;) {
        describe(a_ptrs, a_metas, group, &a);
        describe(b_ptrs, b_metas, group, &b);
        tiles_n = (uint32_t)((b.shape[1] + 255) / 256);
        const uint32_t tiles = (uint32_t)((a.shape[0] + 255) / 256) * tiles_n;
        if (place < tiles) break;
        place -= tiles, ++group;
      }
      describe(c_ptrs, c_metas, group, &c);
      PartitionArg<2> z;
      z.ptr = c.ptr;
      z.shape[0] = c.shape[0], z.shape[1] = c.shape[1];
      z.strides[0] = z.pstrides[0] = c.strides[0], z.strides[1] = z.pstrides[1] = 1;
      z.pshape[0] = z.pshape[1] = 256;
      Ring::run_tile_in(Ring::Stages{xs0, xs1, xs2, ys0a, ys0b, ys1a, ys1b}, z, a, b, a.shape[1], place / tiles_n, place % tiles_n, 0);
      __syncthreads();   // the output bands live in the stages that the next tile refills
    }
  }
};

}  // namespace

extern "C" __global__ void __launch_bounds__(512)
    group_gemm_nt_desc_entry__f16_128x128x64_d2x2_ahead(TensorArg<1> a_ptrs, TensorArg<1> b_ptrs, TensorArg<1> c_ptrs, TensorArg<2> a_metas, TensorArg<2> b_metas,
                                                        TensorArg<2> c_metas, int32_t num_groups, float* partials, uint32_t* counters) {
  GroupAhead::run(a_ptrs, b_ptrs, c_ptrs, a_metas, b_metas, c_metas, num_groups, partials, counters);
}
extern "C" __global__ void __launch_bounds__(512)
    group_gemm_nt_desc_entry__f16_256x256x64_q2x4_ahead(TensorArg<1> a_ptrs, TensorArg<1> b_ptrs, TensorArg<1> c_ptrs, TensorArg<2> a_metas, TensorArg<2> b_metas,
                                                        TensorArg<2> c_metas, int32_t num_groups, float* partials, uint32_t* counters) {
  GroupWide::run(a_ptrs, b_ptrs, c_ptrs, a_metas, b_metas, c_metas, num_groups, partials, counters);
}
