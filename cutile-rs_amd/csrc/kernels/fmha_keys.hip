// Attention forward for launches of few query tiles: the wavefronts of a workgroup share the keys of R x 32 query rows instead of holding
// 32 rows each.
//
// What bounds a short launch is the length of the longest chain, not the work: with 32 rows to a wavefront a query tile walks its keys 64
// at a time, 1.1 us each at D = 128, and 4 heads of 1700 rows are 28 workgroups of the 256-row kernel on 256 compute units.  Here S
// wavefronts take 32 keys each of every S x 32, on their own running maximum, sum and output; at the end the S partial outputs go through
// LDS and every wavefront adds up its share of the columns, in the order of the keys.  Fragments, masks and the softmax are those of Fmha
// (fmha.hip).  us before and here: 4 heads of 1700 rows, causal, D = 128 36.5 and 21; 16 of 1024, D = 64 21 and 13; 16 of 505 12.8 and 7.4; 32 of
// 296, not causal, D = 128 15.5 and 9.1.
//
// FmhaOwnKeys (32 rows; 64 at D = 128): a wavefront has keys of its own, in LDS that no other one reads, and the loop no barrier.  The wavefronts of
// FmhaKeys read common stages, filled through registers behind two barriers a step: 256 keys took 3.2 us of 32 rows at D = 128, here 1.2 alone on the chip
// to 1.7 with all of it at work (a compute unit's 128 KiB of K and V from L2 take 1.1; products 0.4, exponentials and their like 0.5).  On 64 rows a step is 1.6 to 2.2 us where 128 keys took
// 1.5: the bounds of both pipes, of LDS and of L2 are about one each.  us on common stages and here: 8 heads of 17 rows behind 3905 keys 50 and 27, 36 of 222 behind 2641
// 52 and 27; 64 rows: 8 heads of 2000 32 and 25, 24 of 800 20 and 22.  At D = 64, where two workgroups with common stages fit a compute unit, those stay
// for 64 rows (16 heads of 1132 19.9 and 25.0).
//
// Where a round of workgroups leaves compute units idle, several take the keys of one query tile (KeyShares): 27 -> 12.9 us, and 12 heads of 28 rows behind 5078 keys
// 62 on common stages, 33 on own ones, 15.2 on eight workgroups each.  Their results meet in the stream's workspace, past the L2s that the XCDs do not
// share; the last to arrive adds them up in the order of the keys, about 2 us and 0.3 to 0.7 for each.
//
// "halves": two wavefronts to 32 rows on the 128 rows of Fmha's workgroup, for launches of many tiles too.  At D = 64 a 64-key step of Fmha is one
// chain of products, exponentials and products on one wavefront of a SIMD; here two wavefronts (four, with two workgroups to a compute unit)
// have 32 keys each and run across each other's waits: 32 heads of 4096 196 -> 180 us, causal 109 -> 102; 192 of 653 51 -> 47, causal 36 -> 32; 64
// of 430, causal 11.7 -> 10.4.  (At D = 128 the registers leave one workgroup to a compute unit: 32 heads of 2048 92 us where the
// ping-pong kernel takes 61.)
#include <hip/hip_runtime.h>

#include "fmha_common.h"
#include "key_steps.h"
#include "split_k.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kOob = 0x80000000u;   // out of range of every resource made here

// Keys of a query tile dealt to several workgroups (blockIdx.z), `steps` key steps each: where their results meet.
struct KeyShares {
  float* partials;      // [head * query tiles + tile][blockIdx.z]: outputs in the order of the lanes that hold them, then (maximum, sum) a row
  uint32_t* counters;   // one to a (head, query tile), 0 between launches
  int32_t steps;
  int32_t pad;
};

// The results of a query tile's workgroups, added up by the one that arrives last: o, m and l of PASSES x (row, four columns) a lane, o not divided
// by l yet.  False in the workgroups that have no more to do.  The shares are added in the order of their keys, whichever came first.
template <int PASSES, int ROWS_OF, int THREADS>
__device__ __forceinline__ bool add_key_shares(const KeyShares& ks, uint32_t tile, uint32_t share, uint32_t shares, f32x4 (&o)[PASSES], float (&m)[PASSES],
                                               float (&l)[PASSES], const int (&row)[PASSES], bool writes_stats, uint32_t* flag) {
  constexpr uint32_t kOut = PASSES * THREADS * 16, kBytes = kOut + ROWS_OF * 8;
  const uint32_t tid = threadIdx.x;
  const __amdgpu_buffer_rsrc_t part = make_rsrc((unsigned char*)ks.partials + (size_t)tile * gridDim.z * kBytes, kBytes * gridDim.z);
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    gemm::store_partial(o[p], part, share * kBytes + p * (THREADS * 16) + tid * 16);
    if (writes_stats)
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{m[p], l[p]}), part, share * kBytes + kOut + row[p] * 8, 0, gemm::kAgentScope);
  }
  if (!gemm::last_to_arrive(ks.counters + tile, shares, flag)) return false;
  constexpr uint32_t kAtOnce = 4;   // shares whose reads are under way together: past the L2 they take about a microsecond
#pragma unroll
  for (int p = 0; p < PASSES; ++p) o[p] = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, m[p] = -INFINITY, l[p] = 0.0f;
#pragma unroll 1
  for (uint32_t k = 0; k < shares; k += kAtOnce) {
    u32x4 v[kAtOnce][PASSES];
    f32x2 st[kAtOnce][PASSES];   // (maximum, sum)
#pragma unroll
    for (uint32_t i = 0; i < kAtOnce; ++i)
#pragma unroll
      for (int p = 0; p < PASSES; ++p) {
        const bool wanted = k + i < shares;
        const uint32_t at = wanted ? (k + i) * kBytes : 0;
        v[i][p] = __builtin_amdgcn_raw_buffer_load_b128(part, wanted ? tid * 16 : kOob, at + p * (THREADS * 16), gemm::kAgentScope);
        st[i][p] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(part, wanted ? kOut + row[p] * 8 : kOob, at, gemm::kAgentScope));
      }
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      float top = m[p];
#pragma unroll
      for (uint32_t i = 0; i < kAtOnce; ++i) top = fmaxf(top, k + i < shares ? st[i][p][0] : -INFINITY);
      const float use = top == -INFINITY ? 0.0f : top;   // no key seen so far: keep exp2 finite
      const float was = __builtin_amdgcn_exp2f(m[p] - use);
      m[p] = top, l[p] *= was, o[p] *= was;
#pragma unroll
      for (uint32_t i = 0; i < kAtOnce; ++i) {
        const float w = k + i < shares ? __builtin_amdgcn_exp2f(st[i][p][0] - use) : 0.0f;
        const f32x4 t = __builtin_bit_cast(f32x4, v[i][p]);
        l[p] = __builtin_fmaf(st[i][p][1], w, l[p]);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[p][e] = __builtin_fmaf(t[e], w, o[p][e]);
      }
    }
  }
  return true;
}

// Where wavefront w of a workgroup left its partial output: one array after another, or half of them in each of two.
template <int D>
struct Bands {
  unsigned char *first, *second;
  int in_first;
  __device__ __forceinline__ unsigned char* operator[](int w) const { return (w < in_first ? first + w * (32 * D * 4) : second + (w - in_first) * (32 * D * 4)); }
};
template <int D>
struct OneBand {
  unsigned char* first;
  __device__ __forceinline__ unsigned char* operator[](int w) const { return first + w * (32 * D * 4); }
};

// What a lane has of the results of a row block (32 query rows) whose keys S wavefronts share: four columns of PASSES rows.
template <int S, int D>
struct RowShare {
  static constexpr int UNITS = D / 4 / S, ROWS = 64 / UNITS, PASSES = 32 / ROWS;   // 16-byte units of a row to a wavefront, rows at a time
};

// Pass p over the partial outputs and statistics that those wavefronts left in LDS (from wavefront `first` on), added up in the order of a step's keys: wavefront wk its share of the columns.
template <int S, int D, typename BANDS>
__device__ __forceinline__ void merge_pass(const BANDS& bands, const float (*row_max)[32], const float (*row_sum)[32], int first, int wk, int p, f32x4& o, float& m, float& l) {
  using H = RowShare<S, D>;
  const int lane = threadIdx.x & 63, unit = wk * H::UNITS + lane % H::UNITS;
  const int r = p * H::ROWS + lane / H::UNITS;
  float top = -INFINITY;
#pragma unroll
  for (int s = 0; s < S; ++s) top = fmaxf(top, row_max[first + s][r]);
  const float use = top == -INFINITY ? 0.0f : top;
  float sum = 0.0f;
  f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const float w = __builtin_amdgcn_exp2f(row_max[first + s][r] - use);
    sum = __builtin_fmaf(row_sum[first + s][r], w, sum);
    const f32x4 part = *reinterpret_cast<const f32x4*>(bands[first + s] + r * (D * 4) + ((unit ^ (r & 15)) << 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = __builtin_fmaf(part[e], w, t[e]);
  }
  o = t, m = top, l = sum;
}

// Four columns of row `qr`, from `unit` on.
template <typename T>
__device__ __forceinline__ void store_row(const PartitionArg<3>& out, int32_t bh, int32_t q_len, int32_t qr, int unit, const f32x4& o, float l) {
  using E = Elem<T>;
  const float sum = fmaxf(l, 1.0e-8f);   // a row that saw no key: 0 (as in Fmha)
  if (qr < out.shape[1] && qr < q_len) {
    const u32x2 w = {E::pack2(o[0] / sum, o[1] / sum), E::pack2(o[2] / sum, o[3] / sum)};
    *reinterpret_cast<u32x2*>((T*)out.ptr + (int64_t)bh * out.strides[0] + (int64_t)qr * out.strides[1] + unit * 4) = w;
  }
}

// Stores the rows block0 * 32 .. of B row blocks held so, with those of the workgroups that have the tile's other keys.
template <typename T, int B, int S, int D, int TILE_ROWS>
__device__ __forceinline__ void store_rows(const PartitionArg<3>& out, int32_t bh, int32_t q_len, int32_t tile_row0, int block0, int wk, f32x4 (&o)[B * RowShare<S, D>::PASSES],
                                           float (&m)[B * RowShare<S, D>::PASSES], float (&l)[B * RowShare<S, D>::PASSES], const KeyShares& ks, uint32_t tile, uint32_t shares,
                                           uint32_t* flag) {
  using H = RowShare<S, D>;
  constexpr int N = B * H::PASSES;
  const int lane = threadIdx.x & 63, unit = wk * H::UNITS + lane % H::UNITS;
  int row[N];
#pragma unroll
  for (int p = 0; p < N; ++p) row[p] = (block0 + p / H::PASSES) * 32 + p % H::PASSES * H::ROWS + lane / H::UNITS;
  if (!add_key_shares<N, TILE_ROWS, 512>(ks, tile, blockIdx.z, shares, o, m, l, row, wk == 0 && lane % H::UNITS == 0, flag)) return;
#pragma unroll
  for (int p = 0; p < N; ++p) store_row<T>(out, bh, q_len, tile_row0 + row[p], unit, o[p], l[p]);
}

// One workgroup to all keys of a query tile: its launches are those whose tiles are more than half of the compute units.
template <typename T, int R, int S, int STAGES, int D>
struct FmhaKeys {
  using E = Elem<T>;
  using vec8 = typename E::vec8;
  static constexpr int BM = R * 32, BN = S * 32, kWaves = R * S, kThreads = kWaves * 64;
  static constexpr int kUnitsPerRow = D / 8, kTileUnits = BN * kUnitsPerRow, kLoads = kTileUnits / kThreads;
  static constexpr int kTileBytes = BN * D * 2, kStageBytes = 2 * kTileBytes;
  static constexpr int DB = D / 32;
  static constexpr int kOutBytes = 32 * D * 4;        // of a wavefront's partial output
  static constexpr int kLdsBytes = STAGES * kStageBytes > kWaves * kOutBytes ? STAGES * kStageBytes : kWaves * kOutBytes;   // (the partial outputs lie in the stages)
  static_assert(kTileUnits % kThreads == 0 && (D / 4) % S == 0, "equal shares");
  static_assert(D == 64 || D == 128, "swizzles below");

  __device__ static __forceinline__ int k_off(int r, int u) { return r * (D * 2) + ((u ^ (r & (kUnitsPerRow - 1))) << 4); }
  __device__ static __forceinline__ int v_off(int r, int u) {
    constexpr int mask = kUnitsPerRow >= 16 ? 3 : 1;
    return r * (D * 2) + ((u ^ ((r & mask) << 2)) << 4);
  }

  __device__ static __forceinline__ void run(const PartitionArg<3>& out, const TensorArg<4>& q, const TensorArg<4>& k, const TensorArg<4>& v,
                                             float qk_scale, int32_t input_pos, int32_t group_size, int32_t causal, const TileGrid& g, const KeyShares&) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLdsBytes];
    __shared__ float row_max[kWaves][32], row_sum[kWaves][32];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wr = wave / S, wk = wave % S;
    const int l32 = lane & 31, half = lane >> 5, grp = lane >> 4, l16 = lane & 15;

    const int32_t H = q.shape[1];
    int32_t bh, q_tile;
    head_and_tile(g.x, g.y, causal, (uint32_t)group_size, &bh, &q_tile);
    const int32_t batch = bh / H, head = bh % H, kv_head = head / group_size;
    const int32_t q_len = q.shape[2], k_len = k.shape[2];
    const int32_t q0 = q_tile * BM + wr * 32;   // first query row of this wavefront

    const T* qb = (const T*)q.ptr + (int64_t)batch * q.strides[0] + (int64_t)head * q.strides[1];
    const T* kb = (const T*)k.ptr + (int64_t)batch * k.strides[0] + (int64_t)kv_head * k.strides[1];
    const T* vb = (const T*)v.ptr + (int64_t)batch * v.strides[0] + (int64_t)kv_head * v.strides[1];
    const int32_t q_ld = q.strides[2], k_ld = k.strides[2], v_ld = v.strides[2];
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(qb, rows_extent_bytes(q_len, q_ld, D));
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kb, rows_extent_bytes(k_len, k_ld, D));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vb, rows_extent_bytes(k_len, v_ld, D));

    // Qᵀ operand: lane holds query row q0 + l32, d = ks*16 + half*8 .. +7.
    vec8 qf[D / 16];
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const uint32_t off = q0 + l32 < q_len ? (uint32_t)(((int64_t)(q0 + l32) * q_ld + ks * 16 + half * 8) * 2) : kOob;
      qf[ks] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0));
    }
    const int32_t keys = keys_seen((q_tile + 1) * BM, q_len, input_pos, k_len, causal);   // that any row of the workgroup sees
    const int32_t tc = (keys + BN - 1) / BN;

    int ld_row[kLoads], ld_unit[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int c = tid + i * kThreads;
      ld_row[i] = c / kUnitsPerRow, ld_unit[i] = c % kUnitsPerRow;
    }
    u32x4 k_reg[kLoads], v_reg[kLoads];
    auto load_global = [&](int32_t j) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int32_t r = j * BN + ld_row[i];
        k_reg[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, r < k_len ? (uint32_t)(((int64_t)r * k_ld + ld_unit[i] * 8) * 2) : kOob, 0, 0);
        v_reg[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, r < k_len ? (uint32_t)(((int64_t)r * v_ld + ld_unit[i] * 8) * 2) : kOob, 0, 0);
      }
    };
    auto store_lds = [&](int stage) {
      unsigned char* sk = lds + stage * kStageBytes;
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        *reinterpret_cast<u32x4*>(sk + k_off(ld_row[i], ld_unit[i])) = k_reg[i];
        *reinterpret_cast<u32x4*>(sk + kTileBytes + v_off(ld_row[i], ld_unit[i])) = v_reg[i];
      }
    };

    f32x16 o_acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) o_acc[i][e] = 0.0f;
    float m_i = -INFINITY, l_i = 0.0f;
    const float c = qk_scale * kLog2e;
    const int32_t last_visible = (causal ? min(q0 + l32 + input_pos, k_len - 1) : k_len - 1) - half * 4 - wk * 32;   // last key the lane may see
    const int32_t all_see = causal ? min(q0 + input_pos, k_len - 1) : k_len - 1;             // last key that every row of the wavefront sees
    const int32_t any_sees = causal ? min(q0 + 31 + input_pos, k_len - 1) : k_len - 1;       // last key that one of them sees

    if (tc > 0) {
      load_global(0);
      store_lds(0);
    }
    __syncthreads();
    for (int32_t j = 0; j < tc; ++j) {
      const int cur = STAGES == 2 ? j & 1 : 0;
      if (j + 1 < tc) load_global(j + 1);
      const unsigned char* sk = lds + cur * kStageBytes;
      const unsigned char* sv = sk + kTileBytes;
      const int32_t first = j * BN + wk * 32;   // of the wavefront's keys
      if (first <= any_sees) {
        f32x16 s;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks)
          s = E::mfma(*reinterpret_cast<const vec8*>(sk + k_off(wk * 32 + l32, ks * 2 + half)), qf[ks], s);
        // s[e] belongs to key first + (e/4)*8 + half*4 + e%4 and to this lane's query row
        if (first + 31 > all_see) {
          const int32_t lim = last_visible - j * BN;
#pragma unroll
          for (int e = 0; e < 16; ++e) s[e] = ((e >> 2) * 8 + (e & 3)) <= lim ? s[e] : -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[e]);
        mx = max_across_halves(mx);
        constexpr float kSlack = 8.0f;   // the reference point only has to bound the exponents (as in Fmha)
        const float m_cand = fmaxf(m_i, mx * c);
        const bool moved = __builtin_amdgcn_ballot_w64(m_cand > m_i + kSlack) != 0;
        const float m_new = moved ? m_cand : m_i;
        const float m_use = m_new == -INFINITY ? 0.0f : m_new;   // fully masked so far: keep exp2 finite
        float p[16], rs = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], c, -m_use));
          rs += p[e];
        }
        vec8 pf[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const u32x4 w = {E::pack2(p[t * 8 + 0], p[t * 8 + 1]), E::pack2(p[t * 8 + 2], p[t * 8 + 3]), E::pack2(p[t * 8 + 4], p[t * 8 + 5]),
                           E::pack2(p[t * 8 + 6], p[t * 8 + 7])};
          pf[t] = __builtin_bit_cast(vec8, w);
        }
        if (moved) {
          const float alpha = __builtin_amdgcn_exp2f(m_i - m_use);
          l_i *= alpha;
#pragma unroll
          for (int i = 0; i < DB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) o_acc[i][e] *= alpha;
          m_i = m_new;
        }
        l_i += rs;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int db = 0; db < DB; ++db) {
            const int dcol = db * 32 + (grp & 1) * 16 + (l16 & 3) * 4;
            const int kr = wk * 32 + t * 16 + (grp >> 1) * 4 + (l16 >> 2);
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(sv + v_off(kr, dcol >> 3) + (dcol & 7) * 2));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(sv + v_off(kr + 8, dcol >> 3) + (dcol & 7) * 2));
            o_acc[db] = E::mfma(__builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), pf[t], o_acc[db]);
          }
      }
      if (STAGES == 1) __syncthreads();   // everybody has read the stage
      if (j + 1 < tc) store_lds(cur ^ (STAGES - 1));
      __syncthreads();
    }

    // The partial outputs: row l32 of wavefront w at w * kOutBytes, 16-byte unit u of it at u ^ (row & 15).
    l_i = sum_across_halves(l_i);
    if (half == 0) row_max[wave][l32] = m_i, row_sum[wave][l32] = l_i;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {   // d = db*32 + qd*8 + half*4 ..
        const f32x4 w = {o_acc[db][qd * 4 + 0], o_acc[db][qd * 4 + 1], o_acc[db][qd * 4 + 2], o_acc[db][qd * 4 + 3]};
        *reinterpret_cast<f32x4*>(lds + wave * kOutBytes + l32 * (D * 4) + (((db * 8 + qd * 2 + half) ^ (l32 & 15)) << 4)) = w;
      }
    __syncthreads();
    using Share = RowShare<S, D>;
    const OneBand<D> bands{lds};
#pragma unroll
    for (int p = 0; p < Share::PASSES; ++p) {   // (a row's sums leave as soon as they are there: held back for the rows behind them they cost 1 to 2 % of a short launch)
      f32x4 o;
      float m, l;
      merge_pass<S, D>(bands, row_max, row_sum, wr * S, wk, p, o, m, l);
      store_row<T>(out, bh, q_len, q0 + p * Share::ROWS + lane / Share::UNITS, wk * Share::UNITS + lane % Share::UNITS, o, l);
    }
  }
};

// R x 32 query rows, eight wavefronts with keys of their own: wavefront w takes keys 32 (8 j + w) .. + 31 of step j into a stage that no other one reads,
// so nothing in the loop waits for another wavefront.  K of the next step is requested as soon as this one's fragments are in registers, in front of the
// products, and V likewise: a wavefront has nearly always both on their way, a compute unit 100 to 128 KiB at D = 128.
template <typename T, int R, int D>
struct FmhaOwnKeys {
  using E = Elem<T>;
  using vec8 = typename E::vec8;
  static constexpr int BM = R * 32, kWaves = 8, BN = kWaves * 32;
  static constexpr int kUnitsPerRow = D / 8, kSlabBytes = 32 * D * 2, kInstr = kSlabBytes / 1024, kRowsPerInstr = 32 / kInstr;
  static constexpr int DB = D / 32, KS = D / 16, NO = 2 * DB;
  static constexpr bool kQInLds = R * D > 128;   // beside 64 rows of 128 output columns there are no registers for it
  static constexpr int kQBytes = kQInLds ? BM * D * 2 : 16;
  static_assert(D == 64 || D == 128, "swizzles below");

  __device__ static __forceinline__ int k_off(int r, int u) { return r * (D * 2) + ((u ^ (r & (kUnitsPerRow - 1))) << 4); }
  static constexpr int kVMask = kUnitsPerRow >= 16 ? 3 : 1;
  __device__ static __forceinline__ int v_off(int r, int u) { return r * (D * 2) + ((u ^ ((r & kVMask) << 2)) << 4); }

  __device__ static __forceinline__ void run(const PartitionArg<3>& out, const TensorArg<4>& q, const TensorArg<4>& k, const TensorArg<4>& v,
                                             float qk_scale, int32_t input_pos, int32_t group_size, int32_t causal, const TileGrid& g, const KeyShares& shares_of) {
    // K and V apart: the compiler can then tell a refill of one from reads of the other.  The partial outputs lie across both at the end.
    __shared__ __attribute__((aligned(1024))) unsigned char ks_lds[kWaves * kSlabBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char vs_lds[kWaves * kSlabBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char q_lds[kQBytes];
    __shared__ float row_max[kWaves][32], row_sum[kWaves][32];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int l32 = lane & 31, half = lane >> 5, grp = lane >> 4, l16 = lane & 15;

    const int32_t H = q.shape[1];
    int32_t bh, q_tile;
    head_and_tile(g.x, g.y, causal, (uint32_t)group_size, &bh, &q_tile);
    const int32_t batch = bh / H, head = bh % H, kv_head = head / group_size;
    const int32_t q_len = q.shape[2], k_len = k.shape[2], q0 = q_tile * BM;
    const int32_t keys = keys_seen(q0 + BM, q_len, input_pos, k_len, causal);   // that any row sees
    const KeySteps mine = key_steps(keys, BN, shares_of.steps, blockIdx.z, gridDim.z);
    const uint32_t shares = mine.shares, tile = (uint32_t)bh * g.y + (uint32_t)q_tile;
    const int32_t j0 = mine.first, tc = mine.end;   // key steps of this workgroup
    if (blockIdx.z > 0 && j0 >= tc) return;
    const int32_t my_end = min(tc, (keys - wave * 32 + BN - 1) / BN);   // behind this wavefront's last step with a key that any row sees
    static_assert(R <= 2, "a last step has all row blocks, or the second alone");
    const int32_t low_end = R == 1 ? my_end : min(tc, (keys_seen(q0 + 32, q_len, input_pos, k_len, causal) - wave * 32 + BN - 1) / BN);   // the last one with a key that the first 32 rows see

    const T* qb = (const T*)q.ptr + (int64_t)batch * q.strides[0] + (int64_t)head * q.strides[1];
    const T* kb = (const T*)k.ptr + (int64_t)batch * k.strides[0] + (int64_t)kv_head * k.strides[1];
    const T* vb = (const T*)v.ptr + (int64_t)batch * v.strides[0] + (int64_t)kv_head * v.strides[1];
    const int32_t q_ld = q.strides[2], k_ld = k.strides[2], v_ld = v.strides[2];
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(qb, rows_extent_bytes(q_len, q_ld, D));
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kb, rows_extent_bytes(k_len, k_ld, D));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vb, rows_extent_bytes(k_len, v_ld, D));

    unsigned char* const my_k = ks_lds + wave * kSlabBytes;
    unsigned char* const my_v = vs_lds + wave * kSlabBytes;
    // the LDS side of a direct load is lane contiguous: a lane fetches the unit that belongs at its place
    const int lr = lane / kUnitsPerRow, lu = lane % kUnitsPerRow;
    auto fetch_k = [&](int32_t j) {   // keys of step j; past this wavefront's last step and past the last key zeros, which never leave the compute unit
      const int32_t first = j * BN + wave * 32, rows = j < my_end ? k_len - first : 0;
#pragma unroll
      for (int i = 0; i < kInstr; ++i) {
        const int r = i * kRowsPerInstr + lr;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (LDS_PTR(void))(my_k + i * 1024), 16,
                                                 r < rows ? (uint32_t)(((first + r) * k_ld + (lu ^ (r & (kUnitsPerRow - 1))) * 8) * 2) : kOob, 0, 0, 0);
      }
    };
    auto fetch_v = [&](int32_t j) {
      const int32_t first = j * BN + wave * 32, rows = j < my_end ? k_len - first : 0;
#pragma unroll
      for (int i = 0; i < kInstr; ++i) {
        const int r = i * kRowsPerInstr + lr;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (LDS_PTR(void))(my_v + i * 1024), 16,
                                                 r < rows ? (uint32_t)(((first + r) * v_ld + (lu ^ ((r & kVMask) << 2)) * 8) * 2) : kOob, 0, 0, 0);
      }
    };
    // Qᵀ operand of row block b: lane holds query row q0 + 32 b + l32, d = ks*16 + half*8 .. +7.
    vec8 qf[kQInLds ? 1 : R * KS];
    if constexpr (kQInLds) {
      constexpr int kMine = kQBytes / 1024 / kWaves;
#pragma unroll
      for (int i = 0; i < kMine; ++i) {
        const int r = (wave * kMine + i) * kRowsPerInstr + lr;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (LDS_PTR(void))(q_lds + (wave * kMine + i) * 1024), 16,
                                                 q0 + r < q_len ? (uint32_t)(((q0 + r) * q_ld + (lu ^ (r & (kUnitsPerRow - 1))) * 8) * 2) : kOob, 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int n = 0; n < R * KS; ++n) {
        const int32_t r = q0 + n / KS * 32 + l32;
        qf[n] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(rq, r < q_len ? (uint32_t)((r * q_ld + n % KS * 16 + half * 8) * 2) : kOob, 0, 0));
      }
    }
    fetch_k(j0);
    fetch_v(j0);
    if constexpr (kQInLds) {
      __builtin_amdgcn_s_waitcnt(((2 * kInstr) & 15) | (7 << 4) | (15 << 8) | (((2 * kInstr) >> 4) << 14));   // this wavefront's share of Q
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    // Fragment ks of K (or Q) lies at k_base ^ (ks << 5), block db of V at v_base ^ (db << 6): the swizzles are exclusive ors of the unit.  (Formed anew in every step,
    // hidden from the compiler, which would keep all of them in registers.)
    const int k_base = wave * kSlabBytes + k_off(l32, half), q_base = k_off(l32, half);
    const int v_base = wave * kSlabBytes + v_off((grp >> 1) * 4 + (l16 >> 2), (grp & 1) * 2 + ((l16 & 3) >> 1)) + (l16 & 1) * 8;

    f32x16 o_acc[R][DB];
    float m_i[R], l_i[R];
#pragma unroll
    for (int b = 0; b < R; ++b) {
      m_i[b] = -INFINITY, l_i[b] = 0.0f;
#pragma unroll
      for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o_acc[b][i][e] = 0.0f;
    }
    const float c = qk_scale * kLog2e;
    const int32_t all_see = causal ? min(q0 + input_pos, k_len - 1) : k_len - 1;   // last key that every row sees
    constexpr int kWaitOlder = (kInstr & 15) | (7 << 4) | (15 << 8);               // all but the newest kInstr requests have landed
    constexpr int kReadsHome = 15 | (3 << 14) | (7 << 4);                          // LDS reads only

    // a key step of row blocks B0 ..
    auto step = [&](int32_t j, auto from) {
      constexpr int B0 = decltype(from)::value;
      const int32_t first = j * BN + wave * 32;   // of the wavefront's keys
      __builtin_amdgcn_s_waitcnt(kWaitOlder);     // K (V behind it may be on its way)
      __builtin_amdgcn_sched_barrier(0);
      int k_at = k_base, q_at = q_base, v_at = v_base;
      asm volatile("" : "+v"(k_at), "+v"(q_at), "+v"(v_at));
      vec8 kf[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = *reinterpret_cast<const vec8*>(ks_lds + (k_at ^ (ks << 5)));
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(kReadsHome);
      __builtin_amdgcn_sched_barrier(0);
      fetch_k(j + 1);
      __builtin_amdgcn_sched_barrier(0);
      f32x16 s[R];
#pragma unroll
      for (int b = B0; b < R; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[b][e] = 0.0f;
      if constexpr (kQInLds) {
        constexpr int kAhead = 2, kRing = kAhead + 1;   // a read takes longer than the products of one step
        vec8 ring[kRing][R];
        auto read_q = [&](int ks, vec8 (&into)[R]) {
#pragma unroll
          for (int b = B0; b < R; ++b) into[b] = *reinterpret_cast<const vec8*>(q_lds + (q_at ^ (ks << 5)) + b * 32 * (D * 2));
        };
#pragma unroll
        for (int ks = 0; ks < kAhead; ++ks) read_q(ks, ring[ks]);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + kAhead < KS) read_q(ks + kAhead, ring[(ks + kAhead) % kRing]);
#pragma unroll
          for (int b = B0; b < R; ++b) s[b] = E::mfma(kf[ks], ring[ks % kRing][b], s[b]);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int b = B0; b < R; ++b) s[b] = E::mfma(kf[ks], qf[b * KS + ks], s[b]);
      }
      // s[b][e] belongs to key first + (e/4)*8 + half*4 + e%4 and to this lane's query row of block b
      vec8 pf[R][2];
#pragma unroll
      for (int b = B0; b < R; ++b) {
        if (first + 31 > all_see) {
          const int32_t lim = (causal ? min(q0 + b * 32 + l32 + input_pos, k_len - 1) : k_len - 1) - half * 4 - first;   // last key the lane may see
#pragma unroll
          for (int e = 0; e < 16; ++e) s[b][e] = ((e >> 2) * 8 + (e & 3)) <= lim ? s[b][e] : -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[b][e]);
        mx = max_across_halves(mx);
        constexpr float kSlack = 8.0f;   // the reference point only has to bound the exponents (as in Fmha)
        const float m_cand = fmaxf(m_i[b], mx * c);
        const bool moved = __builtin_amdgcn_ballot_w64(m_cand > m_i[b] + kSlack) != 0;
        const float m_new = moved ? m_cand : m_i[b];
        const float m_use = m_new == -INFINITY ? 0.0f : m_new;   // fully masked so far: keep exp2 finite
        float p[16], rs = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][e], c, -m_use));
          rs += p[e];
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const u32x4 w = {E::pack2(p[t * 8 + 0], p[t * 8 + 1]), E::pack2(p[t * 8 + 2], p[t * 8 + 3]), E::pack2(p[t * 8 + 4], p[t * 8 + 5]),
                           E::pack2(p[t * 8 + 6], p[t * 8 + 7])};
          pf[b][t] = __builtin_bit_cast(vec8, w);
        }
        if (moved) {
          const float alpha = __builtin_amdgcn_exp2f(m_i[b] - m_use);
          l_i[b] *= alpha;
#pragma unroll
          for (int i = 0; i < DB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) o_acc[b][i][e] *= alpha;
          m_i[b] = m_new;
        }
        l_i[b] += rs;
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(kWaitOlder);   // V (the next K behind it may be on its way)
      __builtin_amdgcn_sched_barrier(0);
      vec8 vf[NO];
#pragma unroll
      for (int n = 0; n < NO; ++n) {   // step n of Oᵀ: t = n / DB, db = n % DB
        const unsigned char* p = vs_lds + (v_at ^ ((n % DB) << 6)) + (n / DB) * 16 * (D * 2);   // + 8 rows the second half: the same swizzle
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))p);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(p + 8 * (D * 2)));
        vf[n] = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(kReadsHome);
      __builtin_amdgcn_sched_barrier(0);
      fetch_v(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < NO; ++n)
#pragma unroll
        for (int b = B0; b < R; ++b) o_acc[b][n % DB] = E::mfma(vf[n], pf[b][n / DB], o_acc[b][n % DB]);
    };
    int32_t j = j0;
    for (; j < low_end; ++j) step(j, std::integral_constant<int, 0>{});
    // (keys that only the other block's rows see: zero times a value that is not finite would not be zero in the first one.  A branch around the products instead spills 316 bytes a lane)
    if constexpr (R > 1)
      if (j < my_end) step(j, std::integral_constant<int, 1>{});
    __builtin_amdgcn_s_waitcnt(0);   // trailing (zero-filling) fetches must not land in what follows

    // The partial outputs, row block by row block: row l32, 16-byte unit u of it at u ^ (row & 15), in LDS that other wavefronts have done with, too.
    using Share = RowShare<kWaves, D>;
    const Bands<D> bands{ks_lds, vs_lds, kWaves / 2};
    f32x4 o[R * Share::PASSES];
    float m[R * Share::PASSES], l[R * Share::PASSES];
#pragma unroll
    for (int b = 0; b < R; ++b) {
      __syncthreads();
      const float sum = sum_across_halves(l_i[b]);
      if (half == 0) row_max[wave][l32] = m_i[b], row_sum[wave][l32] = sum;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {   // d = db*32 + qd*8 + half*4 ..
          const f32x4 w = {o_acc[b][db][qd * 4 + 0], o_acc[b][db][qd * 4 + 1], o_acc[b][db][qd * 4 + 2], o_acc[b][db][qd * 4 + 3]};
          *reinterpret_cast<f32x4*>(bands[wave] + l32 * (D * 4) + (((db * 8 + qd * 2 + half) ^ (l32 & 15)) << 4)) = w;
        }
      __syncthreads();
#pragma unroll
      for (int p = 0; p < Share::PASSES; ++p) {
        const int at = b * Share::PASSES + p;
        merge_pass<kWaves, D>(bands, row_max, row_sum, 0, wave, p, o[at], m[at], l[at]);
        if (shares == 1) store_row<T>(out, bh, q_len, q0 + b * 32 + p * Share::ROWS + lane / Share::UNITS, wave * Share::UNITS + lane % Share::UNITS, o[at], l[at]);
      }
    }
    if (shares > 1) store_rows<T, R, kWaves, D, BM>(out, bh, q_len, q0, 0, wave, o, m, l, shares_of, tile, shares, reinterpret_cast<uint32_t*>(ks_lds));
  }
};

}  // namespace

#define FMHA_KEYS_KERNEL(NAME, KERNEL)                                                                                              \
  extern "C" __global__ void __launch_bounds__(512)                                                                               \
      fmha_entry__##NAME(PartitionArg<3> out, TensorArg<4> q, TensorArg<4> k, TensorArg<4> v, float qk_scale, int32_t input_pos,   \
                         int32_t query_group_size, int32_t causal, TileGrid g, KeyShares shares) {                                \
    KERNEL::run(out, q, k, v, qk_scale, input_pos, query_group_size, causal, g, shares);                                           \
  }
#define FMHA_KEYS_SEQ_KERNEL(NAME, KERNEL)                                                                                          \
  extern "C" __global__ void __launch_bounds__(512)                                                                               \
      fmha_seq_entry__##NAME(PartitionArg<3> out, TensorArg<4> q, TensorArg<4> k, TensorArg<4> v, float qk_scale,                  \
                             const uint32_t* position_start, int32_t kv_len_from_position, int32_t query_group_size,              \
                             int32_t causal, TileGrid g, KeyShares shares) {                                                      \
    const int32_t pos = (int32_t)min(position_start[0], 0x3fffffffu);                                                              \
    TensorArg<4> kk = k, vv = v;                                                                                                   \
    if (kv_len_from_position) kk.shape[2] = vv.shape[2] = min(min(k.shape[2], v.shape[2]), pos + 1);                               \
    KERNEL::run(out, q, kk, vv, qk_scale, pos, query_group_size, causal, g, shares);                                               \
  }
// rows, wavefronts to 32 of them, stages, D
template <typename T> using Rows32D128 = FmhaOwnKeys<T, 1, 128>;
template <typename T> using Rows32D64 = FmhaOwnKeys<T, 1, 64>;
template <typename T> using Rows64D128 = FmhaOwnKeys<T, 2, 128>;
template <typename T> using Rows64D128Few = FmhaKeys<T, 2, 4, 2, 128>;
template <typename T> using Rows64D64 = FmhaKeys<T, 2, 4, 2, 64>;
template <typename T> using Rows128D64 = FmhaKeys<T, 4, 2, 2, 64>;
FMHA_KEYS_KERNEL(bf16_32x256x128_keys, Rows32D128<__bf16>)
FMHA_KEYS_KERNEL(f16_32x256x128_keys, Rows32D128<_Float16>)
FMHA_KEYS_KERNEL(bf16_32x256x64_keys, Rows32D64<__bf16>)
FMHA_KEYS_KERNEL(f16_32x256x64_keys, Rows32D64<_Float16>)
FMHA_KEYS_KERNEL(bf16_64x128x128_keys, Rows64D128<__bf16>)
FMHA_KEYS_KERNEL(f16_64x128x128_keys, Rows64D128<_Float16>)
FMHA_KEYS_KERNEL(bf16_few_64x128x128_keys, Rows64D128Few<__bf16>)
FMHA_KEYS_KERNEL(f16_few_64x128x128_keys, Rows64D128Few<_Float16>)
FMHA_KEYS_KERNEL(bf16_64x128x64_keys, Rows64D64<__bf16>)
FMHA_KEYS_KERNEL(f16_64x128x64_keys, Rows64D64<_Float16>)
FMHA_KEYS_KERNEL(bf16_128x64x64_halves, Rows128D64<__bf16>)
FMHA_KEYS_KERNEL(f16_128x64x64_halves, Rows128D64<_Float16>)
FMHA_KEYS_SEQ_KERNEL(f16_32x256x128_keys, Rows32D128<_Float16>)
FMHA_KEYS_SEQ_KERNEL(f16_32x256x64_keys, Rows32D64<_Float16>)
FMHA_KEYS_SEQ_KERNEL(f16_64x128x128_keys, Rows64D128<_Float16>)
FMHA_KEYS_SEQ_KERNEL(f16_few_64x128x128_keys, Rows64D128Few<_Float16>)
FMHA_KEYS_SEQ_KERNEL(f16_64x128x64_keys, Rows64D64<_Float16>)
FMHA_KEYS_SEQ_KERNEL(f16_128x64x64_halves, Rows128D64<_Float16>)
