// Attention forward for launches of few query tiles: the wavefronts of a workgroup share the keys of R x 32 query rows instead of holding
// 32 rows each.
//
// What bounds a short launch is the length of the longest chain, not the work: with 32 rows to a wavefront a query tile walks its keys 64
// at a time, 1.1 us each at D = 128, and 4 heads of 1700 rows are 28 workgroups of the 256-row kernel on 256 compute units.  Here S
// wavefronts take 32 keys each of every S x 32, on their own running maximum, sum and output; at the end the S partial outputs go through
// LDS and every wavefront adds up its share of the columns, in the order of the keys.  Fragments, masks and the softmax are those of Fmha
// (fmha.hip).  K and V wait in registers for the stage to be free (STAGES = 1), or go to the other one (STAGES = 2).
// Now a step is bound by the reads of K and V, which every 32 (64) rows repeat: 128 KiB through a compute unit's vector cache at 64 bytes a
// clock are 0.9 of the 2.4 us that 256 keys take at D = 128, the rest their latency and the barriers.  us before and here: 4 heads of 1700
// rows, causal, D = 128 36.5 and 23.4; 16 of 1024, D = 64 21 and 13; 16 of 505 12.8 and 7.4; 32 of 296, not causal, D = 128 15.5 and 11.4.
//
// "halves": two wavefronts to 32 rows on the 128 rows of Fmha's workgroup, for launches of many tiles too.  At D = 64 a 64-key step of Fmha is one
// chain of products, exponentials and products on one wavefront of a SIMD; here two wavefronts (four, with two workgroups to a compute unit)
// have 32 keys each and run across each other's waits: 32 heads of 4096 196 -> 180 us, causal 109 -> 102; 192 of 653 51 -> 47, causal 36 -> 32; 64
// of 430, causal 11.7 -> 10.4.  (At D = 128 the registers leave one workgroup to a compute unit: 32 heads of 2048 92 us where the
// ping-pong kernel takes 61.)
#include <hip/hip_runtime.h>

#include "fmha_common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T, int R, int S, int STAGES, int D>
struct FmhaKeys {
  using E = Elem<T>;
  using vec8 = typename E::vec8;
  static constexpr int BM = R * 32, BN = S * 32, kWaves = R * S, kThreads = kWaves * 64;
  static constexpr int kUnitsPerRow = D / 8, kTileUnits = BN * kUnitsPerRow, kLoads = kTileUnits / kThreads;
  static constexpr int kTileBytes = BN * D * 2, kStageBytes = 2 * kTileBytes;
  static constexpr int DB = D / 32;
  static constexpr int kOutUnits = D / 4;             // 16-byte units of a partial output row
  static constexpr int kOutBytes = 32 * D * 4;        // of a wavefront's partial output
  static constexpr int kLdsBytes = STAGES * kStageBytes > kWaves * kOutBytes ? STAGES * kStageBytes : kWaves * kOutBytes;   // (the partial outputs lie in the stages)
  static_assert(kTileUnits % kThreads == 0 && kOutUnits % S == 0, "equal shares");
  static_assert(D == 64 || D == 128, "swizzles below");

  __device__ static __forceinline__ int k_off(int r, int u) { return r * (D * 2) + ((u ^ (r & (kUnitsPerRow - 1))) << 4); }
  __device__ static __forceinline__ int v_off(int r, int u) {
    constexpr int mask = kUnitsPerRow >= 16 ? 3 : 1;
    return r * (D * 2) + ((u ^ ((r & mask) << 2)) << 4);
  }

  __device__ static __forceinline__ void run(const PartitionArg<3>& out, const TensorArg<4>& q, const TensorArg<4>& k, const TensorArg<4>& v,
                                             float qk_scale, int32_t input_pos, int32_t group_size, int32_t causal, const TileGrid& g) {
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
    constexpr uint32_t kOob = 0x80000000u;

    // Qᵀ operand: lane holds query row q0 + l32, d = ks*16 + half*8 .. +7.
    vec8 qf[D / 16];
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const uint32_t off = q0 + l32 < q_len ? (uint32_t)(((int64_t)(q0 + l32) * q_ld + ks * 16 + half * 8) * 2) : kOob;
      qf[ks] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0));
    }
    const int32_t keys = causal ? min(input_pos + (q_tile + 1) * BM, k_len) : k_len;   // that any row of the workgroup sees
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
    // wavefront (wr, wk) adds up units [wk * UNITS, ..) of the 32 rows, in the order of the keys of a step
    constexpr int UNITS = kOutUnits / S, ROWS = 64 / UNITS;   // rows at a time
    const int unit = wk * UNITS + lane % UNITS;
#pragma unroll
    for (int pass = 0; pass < 32 / ROWS; ++pass) {
      const int row = pass * ROWS + lane / UNITS;
      float m = -INFINITY;
#pragma unroll
      for (int s = 0; s < S; ++s) m = fmaxf(m, row_max[wr * S + s][row]);
      const float m_use = m == -INFINITY ? 0.0f : m;
      float l = 0.0f;
      f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const float w = __builtin_amdgcn_exp2f(row_max[wr * S + s][row] - m_use);
        l = __builtin_fmaf(row_sum[wr * S + s][row], w, l);
        const f32x4 part = *reinterpret_cast<const f32x4*>(lds + (wr * S + s) * kOutBytes + row * (D * 4) + ((unit ^ (row & 15)) << 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(part[e], w, o[e]);
      }
      l = fmaxf(l, 1.0e-8f);   // a row that saw no key: 0 (as in Fmha)
      const int32_t qr = q0 + row;
      if (qr < out.shape[1] && qr < q_len) {
        const u32x2 w = {E::pack2(o[0] / l, o[1] / l), E::pack2(o[2] / l, o[3] / l)};
        *reinterpret_cast<u32x2*>((T*)out.ptr + (int64_t)bh * out.strides[0] + (int64_t)qr * out.strides[1] + unit * 4) = w;
      }
    }
  }
};

}  // namespace

#define FMHA_KEYS_KERNEL(NAME, T, R, S, STAGES, D)                                                                                  \
  extern "C" __global__ void __launch_bounds__(R * S * 64)                                                                        \
      fmha_entry__##NAME(PartitionArg<3> out, TensorArg<4> q, TensorArg<4> k, TensorArg<4> v, float qk_scale, int32_t input_pos,   \
                         int32_t query_group_size, int32_t causal, TileGrid g) {                                                  \
    FmhaKeys<T, R, S, STAGES, D>::run(out, q, k, v, qk_scale, input_pos, query_group_size, causal, g);                             \
  }
#define FMHA_KEYS_SEQ_KERNEL(NAME, T, R, S, STAGES, D)                                                                              \
  extern "C" __global__ void __launch_bounds__(R * S * 64)                                                                        \
      fmha_seq_entry__##NAME(PartitionArg<3> out, TensorArg<4> q, TensorArg<4> k, TensorArg<4> v, float qk_scale,                  \
                             const uint32_t* position_start, int32_t kv_len_from_position, int32_t query_group_size,              \
                             int32_t causal, TileGrid g) {                                                                        \
    const int32_t pos = (int32_t)min(position_start[0], 0x3fffffffu);                                                              \
    TensorArg<4> kk = k, vv = v;                                                                                                   \
    if (kv_len_from_position) kk.shape[2] = vv.shape[2] = min(min(k.shape[2], v.shape[2]), pos + 1);                               \
    FmhaKeys<T, R, S, STAGES, D>::run(out, q, kk, vv, qk_scale, pos, query_group_size, causal, g);                                 \
  }
FMHA_KEYS_KERNEL(bf16_32x256x128_keys, __bf16, 1, 8, 1, 128)
FMHA_KEYS_KERNEL(f16_32x256x128_keys, _Float16, 1, 8, 1, 128)
FMHA_KEYS_KERNEL(bf16_32x256x64_keys, __bf16, 1, 8, 1, 64)
FMHA_KEYS_KERNEL(f16_32x256x64_keys, _Float16, 1, 8, 1, 64)
FMHA_KEYS_KERNEL(bf16_64x128x128_keys, __bf16, 2, 4, 2, 128)
FMHA_KEYS_KERNEL(f16_64x128x128_keys, _Float16, 2, 4, 2, 128)
FMHA_KEYS_KERNEL(bf16_64x128x64_keys, __bf16, 2, 4, 2, 64)
FMHA_KEYS_KERNEL(bf16_128x64x64_halves, __bf16, 4, 2, 2, 64)
FMHA_KEYS_KERNEL(f16_64x128x64_keys, _Float16, 2, 4, 2, 64)
FMHA_KEYS_KERNEL(f16_128x64x64_halves, _Float16, 4, 2, 2, 64)
FMHA_KEYS_SEQ_KERNEL(f16_32x256x128_keys, _Float16, 1, 8, 1, 128)
FMHA_KEYS_SEQ_KERNEL(f16_32x256x64_keys, _Float16, 1, 8, 1, 64)
FMHA_KEYS_SEQ_KERNEL(f16_64x128x128_keys, _Float16, 2, 4, 2, 128)
FMHA_KEYS_SEQ_KERNEL(f16_64x128x64_keys, _Float16, 2, 4, 2, 64)
FMHA_KEYS_SEQ_KERNEL(f16_128x64x64_halves, _Float16, 4, 2, 2, 64)
