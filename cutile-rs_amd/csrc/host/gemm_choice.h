// Which GEMM kernel a launch takes from its extents, where the shape classes of the tuning records are too coarse:
// few rows, outputs of fewer 256 x 256 tiles than compute units (or of a few more), and rows off 16-byte boundaries.
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>

namespace cutile {

struct GemmShape {
  const char* dtype;       // the table's name of the operand / output types: bf16, f16, bf16f32
  int64_t m, n;            // outputs the launch covers
  int64_t y_cols;          // columns of y (a strip or a tile of the gemm_small.hip kernels must lie inside them)
  int32_t k;
  bool aligned;            // rows on 16-byte boundaries, whole output covered: the ring kernels can take it
  bool x_aligned;          // the rows of x are
  bool own_tile;           // the partition's tile has kernels of its own
  bool whole_k;            // K in whole tiles of 64 that both operands have, columns of z in units of 8: the wider tiles can take it
};

// Output tiles of bm x bn of a launch.
inline uint64_t tiles_of(int64_t m, int64_t n, int bm, int bn) { return (uint64_t)((m + bm - 1) / bm) * (uint64_t)((n + bn - 1) / bn); }

// The ring kernels and those of four or five whole stages (gemm_tiles.hip).  One K tile of a launch that fills few compute units costs
// `few` us, of one that fills all of them `all` us (operands through the same L2s, and the clock), and a round of workgroups `ends` us besides.
struct RingTile {
  const char* kernel;
  int bm, bn;
  double few, all, ends;
};
// Least squares over 170 products of 65 to 5000 rows, f16 and bf16, operands from memory, every kernel with K unshared and shared by
// 2 to 8 workgroups (3800 times; 5 to 8 % rms).  Over those sizes the kernel that this prices lowest takes 1.02 times the best one's time.
constexpr RingTile kRingTiles[] = {{"256x256x64_q2x4", 256, 256, 1.03, 1.36, 8.05}, {"192x256x64_q2x4", 192, 256, 0.82, 1.08, 7.2}, {"256x128x64_q4x2", 256, 128, 0.62, 0.865, 5.95},
                                   {"128x256x64_q2x4", 128, 256, 0.62, 0.845, 5.7}, {"192x128x64_q2x2", 192, 128, 0.44, 0.72, 4.5}, {"128x128x64_q2x2", 128, 128, 0.325, 0.55, 4.2}};
// A K tile on 192 x 192 (the stages of 192 x 256), by its share of a wide tile's products: 7 x 36 wide and 7 x 15 narrow tiles of K = 4608 144 us
// priced, 152 measured; 5 x 51 and 5 x 27 of 5120 161, 172; one width 156 and 172 priced, 161 and 179 measured.
constexpr double kNarrowFew = 0.66, kNarrowAll = 0.86, kNarrowEnds = 6.2;
// Wider tiles (gemm_wide.h), priced as above: least squares over 420 products of 200 to 1100 tiles of 192 x 256, K 576 to 14336 (3 to 4 % rms), by 1.08, which is what the
// times of the tiles above were over their prices in those products (median).  Of the 420 they are picked in 138, 0.80 to 1.02 of the other tiles' time, 0.91 in the mean.
struct WideTile {
  const char* member;
  int bm, bn;
  double few, all, ends;
};
constexpr WideTile kWideTiles[] = {{"+w192x320", 192, 320, 0.94, 1.51, 7.1}, {"+w192x384", 192, 384, 1.02, 1.65, 8.5}, {"+w192x448", 192, 448, 1.14, 1.90, 9.3}, {"+w256x320", 256, 320, 1.09, 1.84, 9.4}};
// Workgroups that share a tile: each stores its partial tile, and the last one reads them all.  us a value of one output tile, and of all of them.
constexpr double kShareEach = 4.2e-5, kShareAll = 1.0e-6, kShareOnce = 0.7;
// The one that a kernel of that tile is, by the tile shape and by the marker of these kernels in its name.
inline const RingTile* ring_tile(const char* variant, int bm, int bn) {
  if (bm == 0 || strstr(variant, "x64_q") == nullptr) return nullptr;
  for (const RingTile& r : kRingTiles)
    if (r.bm == bm && r.bn == bn) return &r;
  return nullptr;
}
struct RingPlan {
  uint32_t splits;   // workgroups that share the K tiles of an output tile
  bool two;          // 128 x 128: two workgroups to a compute unit, on the ring (K unshared)
  double us;
  uint32_t wide = 0, narrow = 0;   // columns of tiles, where those of 192 columns stand beside the ones of 256
  const WideTile* by = nullptr;    // these tiles instead
};
// What the launch costs with the best number of workgroups to an output tile; as priced and as launched.  `partial_bytes` = room for partial tiles, 0: K is not shared.
// `wide_tiles`: a launch by the name of 192 x 256 may be on wider ones.
inline RingPlan ring_plan(const RingTile& r, int64_t m, int64_t n, int32_t k, int cus, uint64_t partial_bytes, bool wide_tiles = false) {
  const uint64_t t = tiles_of(m, n, r.bm, r.bn);
  const int64_t kt = (k + 63) / 64;
  RingPlan best{1, false, 1e30};
  for (uint32_t s : {1u, 2u, 3u, 4u, 6u, 8u}) {
    if (s > 1 && (t * s > (uint64_t)cus || kt < 4 * s || t * s * (uint64_t)(r.bm * r.bn * 4) > partial_bytes)) break;
    const uint64_t g = t * s, rest = g % cus;
    const double us = (double)((kt + s - 1) / s) * ((double)(g / cus) * r.all + (rest ? r.few + (r.all - r.few) * (double)rest / cus : 0.0)) +
                      r.ends * (double)((g + cus - 1) / cus) + (s > 1 ? kShareOnce + (kShareEach * s + kShareAll * (double)g) * (r.bm * r.bn) : 0.0);
    if (us < best.us * 0.98) best = {s, false, us};
  }
  if (r.bm == 192 && r.bn == 256 && t > (uint64_t)cus && t < 2 * (uint64_t)cus) {
    // A second round that is not full: a wide tile to each compute unit first, then narrow ones.
    const int64_t rows = (m + r.bm - 1) / r.bm, wide = cus / rows, narrow = (n - wide * 256 + 191) / 192;
    if (wide > 0 && narrow > 0 && rows * (wide + narrow) <= 2 * cus) {
      const double rest = (double)(rows * (wide + narrow) - cus) / cus;
      const double us = (double)kt * (r.all + kNarrowFew + (kNarrowAll - kNarrowFew) * rest) + r.ends + kNarrowEnds;
      if (us < best.us * 0.98) best = {1, false, us, (uint32_t)wide, (uint32_t)narrow};
    }
  }
  if (wide_tiles && r.bm == 192 && r.bn == 256)
    for (const WideTile& w : kWideTiles) {
      const uint64_t g = tiles_of(m, n, w.bm, w.bn), rest = g % cus;
      const double us = (double)kt * ((double)(g / cus) * w.all + (rest ? w.few + (w.all - w.few) * (double)rest / cus : 0.0)) + w.ends * (double)((g + cus - 1) / cus);
      if (us < best.us * 0.98) best = {1, false, us, 0, 0, &w};
    }
  if (r.bm == 128 && r.bn == 128) {
    // two workgroups to a compute unit, each at half its pace as soon as there are more than compute units (1623 x 2944 x
    // 14016 f16, 299 tiles: 214 us, 192 x 128 tiles 151; 619 x 8832 x 7552 bf16, 345 tiles: 137, 256 x 128 tiles 90)
    const uint64_t slots = 2 * (uint64_t)cus, rest = t % slots;
    const double part = rest == 0 ? 0.0 : rest <= (uint64_t)cus ? 0.475 + 0.125 * (double)rest / cus : 1.05 + 0.02 * (double)(rest - cus) / cus;
    const double us = (double)kt * ((double)(t / slots) * 1.07 + part) + 4.5 * (double)((t + slots - 1) / slots);
    if (us < best.us * 1.04) best = {1, true, us};
  }
  return best;
}

// 16-bit weights of this size are not found in the caches by the launch that reads them next (gemm_thin.h).
inline bool streamed_past_caches(int64_t n, int32_t k) { return n * k * 2 >= (96ll << 20); }
// K splits of a thin launch: about one workgroup per compute unit, and at least one 64-row step for each of its 8 wavefronts as far as 8 splits, two beyond
// (operands from memory, us with two steps and with one: 1 x 64 x 4096 6.6, 5.2; 1 x 1024 x 2048 7.5, 5.8; 1 x 2560 x 2560 10.5, 6.7; 20 x 512 x 4096
// 8.6, 6.6; 30 x 2560 x 2560 13.5, 8.0; 40 x 3000 x 3001 22.2, 16.7; 48 x 2048 x 4096 12.0, 10.2).  Strips of 128 columns, which are many: two steps.
// `aligned`: rows on 16-byte boundaries.  Off them a step takes longer and sharing pays sooner (K in 1 and in 2: 16 x 7552 x 1856 7.7,
// 8.4; 8 x 5730 x 1852 8.4, 7.6).  Over 917 products of 1 to 128 rows (K 1024 to 16384) the split chosen here takes 1.015 of the best one's time in the mean, and
// at most 1.08 of what two steps to a wavefront take; the three rules that `aligned` selects take their part of them from as much as 1.21 to 1.04.
inline uint32_t thin_splits(uint64_t blocks, int32_t k, int cus, int rows, int cols, bool aligned) {
  blocks = std::max<uint64_t>(blocks, 1);
  const int64_t halves = k / (64 * 8 * 2), n = (int64_t)blocks;
  // Beyond a quarter of the compute units a short K gains nothing from one step to a wavefront (us in 1 and more: 8 x 5632 x 1536 6.5, 7.2; 7 x 4288 x 2048
  // in 2 and 4 6.7, 7.4; 22 x 7616 x 1600 7.7, 8.6; 120 x 3648 x 1088 9.0, 9.6) but where three shares of the strips lie evenly over the XCDs (24 x 5120 x 1536 8.3, 7.2).
  const bool short_k = aligned && n * 9 > 2 * cus && (rows == 64 ? k < 1152 : k < 2240 && !(n % 8 == 0 && n * 3 <= cus && k >= 1536));
  const int64_t most = cols == 128 || (rows == 16 && k < 1536) || short_k ? halves : std::min<int64_t>(k / (64 * 8), std::max<int64_t>(8, halves));   // (1 x 808 x 1305 5.6, 5.9)
  int64_t best = std::max<int64_t>(1, std::min<int64_t>(cus / n, most));
  if (aligned && best * n * 2 > cus) {   // no more of them than the longest share asks for, if they come out even (12 x 3072 x 3072 in 3, 5 and 6: 7.2, 7.9, 7.9 us)
    const int64_t steps = k / 64, longest = (steps + 8 * best - 1) / (8 * best), even = steps / std::max<int64_t>(8 * longest, 1);
    if (even > 0 && even * 8 * longest == steps) best = even;
  }
  if (rows > 16 || cols == 128) return (uint32_t)best;   // (a second workgroup to a compute unit: 30 x 6144 x 4096 17.1, 19.1; 30 x 3072 x 2048 7.8, 8.5)
  // Where one workgroup to a compute unit leaves some of them idle, two or three (at most 8 to a strip), if the longest share of K, in whole
  // steps of its wavefronts, is shorter for it, or no longer where the last round is nearly full (1 x 4480 x 4096 in 3 and 8, 560 workgroups: 8.9, 10.1; 3 x 6080 x 3072
  // in 2 and 6, 570: 9.1, 10.0) - and shorter by a tenth where K would not be shared at all, of 2560 and more (3 x 10304 x 2496 in 1 and 3: 11.5, 11.9).
  // (4096 x 6144, 96 strips, in 2, 5 and 8: 13.9, 14.3, 13.0 us; 4096 x 11008, 172, in 1 and 4: 19.7, 18.2; 5120 x 5120, 80, in 3 and 6: 15.4, 13.9;
  // 1024 x 14000, 219, in 1 and 2: 7.5, 9.0).
  if (aligned && best == 1 && k < 2560) return 1;
  auto share = [&](int64_t s, int64_t deep) { return (double)(deep * ((k + s * 512 - 1) / (s * 512))); };   // steps of a wavefront, workgroup after workgroup
  const bool alone = best == 1;
  if (best * n <= cus && best < most)
    for (int64_t deep = 2; deep <= 3; ++deep) {
      const int64_t s = std::min<int64_t>({deep * cus / n, most, 8});
      if (s <= best || s * n <= (deep - 1) * cus) continue;
      const double was = share(best, (best * n + cus - 1) / cus) * (best == 1 ? 0.9 : 1.0), is = share(s, deep);
      if (is < was || (is == was && (!aligned || alone || s * n * 10 >= 9 * deep * cus))) best = s;
    }
  return (uint32_t)best;
}
// K splits of a staged launch, as priced below and as launched: 64 x 64 tiles only (64 x 128 with two splits and with none: 336 x
// 2575 x 1350 21.9, 17.8 us; 586 x 1537 x 1527 25.8, 20.4; 193 x 867 x 1070 17.0, 15.5; 130 x 1001 x 1030 15.8, 14.4), up to two workgroups per compute unit, at least 8 K tiles each (1262 x 128 x 16128, 40 tiles: 99, 54, 40, 32,
// 30 us with 1, 2, 3, 4, 8 splits; 128 x 4096 x 4096, 128 tiles: 40, 28.5, 28.0, 28.2, 47).
inline uint32_t staged_splits(int bm, int bn, uint64_t blocks, int32_t k, int cus) {
  if (bm != 64 || bn != 64) return 1;
  return (uint32_t)std::max<int64_t>(1, std::min<int64_t>({(int64_t)(2 * (uint64_t)cus / std::max<uint64_t>(blocks, 1)), k / (64 * 8), 8}));
}

// f32: strips of 64 columns by 16, 32 or 64 rows (gemm_f32.hip).  ns a K position of a strip with the compute unit to itself (the chip then
// does 83, 88 and 94 TFLOP/s on the matrix cores, of 157 nominal), us of start and output; least squares over 119 products of 1 to 4096
// rows, K shared by 1 to 16 workgroups (10 to 12 % rms; the strip and split priced lowest take 1.02 times the best ones' time).  The any-layout kernel
// that ran before: 3 x 2160 x 2208 338 us, strips 9.9; 567 x 64 x 378 49, 6.2; 403 x 1232 x 5728 1055, 119; 107 x 364 x 6461 1345, 19.
struct F32Strip {
  const char* kernel;
  int rows;
  double k, each;   // `each`: ns a value of an output strip for each of the workgroups that share its K
};
constexpr F32Strip kF32Strips[] = {{"strip16x64", 16, 6.35, 0.23}, {"strip32x64", 32, 11.8, 0.11}, {"strip64x64", 64, 22.3, 0.055}};
inline const F32Strip* f32_strip(int rows) {
  for (const F32Strip& r : kF32Strips)
    if (r.rows == rows) return &r;
  return nullptr;
}
struct F32Plan {
  uint32_t splits;
  double us;
};
inline F32Plan f32_plan(const F32Strip& r, int64_t m, int64_t n, int32_t k, int cus, uint64_t partial_bytes) {
  const uint64_t t = tiles_of(m, n, r.rows, 64);
  F32Plan best{1, 1e30};
  for (uint32_t s : {1u, 2u, 4u, 8u, 16u}) {
    if (s > 1 && (t * s > 2 * (uint64_t)cus || k < 128 * (int64_t)s || t * s * (uint64_t)(r.rows * 64 * 4) > partial_bytes)) break;
    const uint64_t g = t * s;
    const double rounds = (double)std::max<uint64_t>(1, (g + cus - 1) / cus), values = r.rows * 64;
    const double us = (double)k / s * r.k * 1e-3 * rounds + 2.1 * (rounds + 1) + (s > 1 ? 0.8 + (r.each * s * 1e-3 + 4e-6 * (double)g / cus) * values : 0.0);
    if (us < best.us * 0.98) best = {s, us};
  }
  return best;
}

// The same for 64 x 64 tiles of aligned rows with a workspace, priced by the number of workgroups: up to one to a compute unit, which shares no K where
// that many tiles are there already (us, K shared by as many as staged_splits says or on 128 x 128 tiles, and here: 272 x 2176 x 1536 17.3, 13.0, both from memory; 374 x 1344 x 1024 9.7, 8.1 from the caches).  Least squares over 1133
// times of 260 products of 66 to 1800 rows, K shared by 1 to 8 (6.5 % rms); without the floor below, over the 231 of them that are not strips, the kernel and split chosen take 0.98 of the time
// before, 41 are chosen otherwise, 0.88 in the mean, one of them slower (706 x 448 x 8512 18.8, 19.5; with a rule that follows the prices alone 80, of which 5 by 2 to 12 %).
struct StagedPlan {
  uint32_t splits;
  double us;
};
inline StagedPlan staged_plan(int64_t m, int64_t n, int32_t k, int cus) {
  const int64_t t = (int64_t)tiles_of(m, n, 64, 64), kt = (k + 63) / 64;
  const uint32_t even = staged_splits(64, 64, (uint64_t)t, k, cus);
  StagedPlan best{1, 0.0};
  double least = 1e30;
  for (uint32_t s = 1; s <= 8; ++s) {
    if (s > 1 && s != even && (kt < 4 * s || t * s > 2 * cus)) continue;
    const double x = (double)(t * s) / cus, fitted = x <= 1.0 ? 0.214 + 0.046 * x : 0.368 + 0.163 * (x - 1.0);
    // (fitted with operands that the caches still hold; from memory a K tile of an unshared tile is 0.36 us however few there are, and the kernels it is
    // compared with are 8 % slower.  At 0.30 no one of 56 products from memory loses by more than 1.3 %; unpriced 174 x 2048 x 2048 14.7 -> 16.1 us, 230 x 2560 x 2560 17.6 ->
    // 19.6, while 272 x 2176 x 1536 17.3 -> 13.0, 230 x 3072 x 1024 12.9 -> 10.3 stay)
    const double rate = s == 1 ? std::max(fitted, 0.30) : fitted;
    const double us = 4.47 + (double)((kt + s - 1) / s) * rate + (s > 1 ? 2.04 + 0.11 * s + 1.88e-6 * (double)(m * n * (int64_t)s) : 0.0);
    if (us * (s == even ? 0.9 : 1.0) < least) least = us * (s == even ? 0.9 : 1.0), best = {s, us};
  }
  return best;
}

struct GemmChoice {
  char variant[48] = "";   // "": the partition's own tile (tuning record, then the table's order)
  bool needs_room = false; // the choice counts on room for partial sums: without it the kernel is to be chosen again
  const RingTile* ring = nullptr;    // the kernel chosen, if it is one of these, and its plan
  RingPlan ring_plan{};
  const F32Strip* strip = nullptr;
  F32Plan strip_plan{};
  uint32_t staged = 0;               // K splits of a staged kernel, where they are not staged_splits'
};

// Register-staged tiles and their prices (choose_gemm): us per K tile, alone on a compute unit and for each of several; us of start and output, paid by every round
// of workgroups; the share by which x rows off 16-byte boundaries lengthen it all; us of shared K, and for each value of the partial sums.  (Tables are
// constants of this file: a static of an inline function is one object for all builds of the library in a process, whichever is loaded first.)
struct StagedTile {
  const char* kernel;
  int bm, bn, per_cu;
  struct Prices { double one, more, ends, x, split, sum; } any, aligned;
};
// Rows off 16-byte boundaries, least squares over 140 products, operands from memory, every tile timed (10 to 13 % rms): over them the tile priced lowest takes
// 1.005 times the best one's time, over 400 more with K up to 700 1.004.  Rows on them, 520 products of 65 to 2500 rows and up to 128 tiles of 128 x 128, with and without a workspace (4 to 6 %
// rms), 64 x 64 tiles 2 % dearer than fitted, as ring tiles of that price are the better ones, and the larger ones 20 % (805 x 1792 x 3264 22.2 us, ring 18.5).
constexpr StagedTile kStaged[] = {{"staged256x256", 256, 256, 1, {1.14, 0, 12.7, 0.126, 0, 0}, {}},
                                  {"staged256x128", 256, 128, 1, {0.77, 0, 8.2, 0.142, 0, 0}, {}},
                                  {"staged128x128", 128, 128, 2, {0.50, 0.52, 6.7, 0.139, 0, 0}, {0.56, 0.28, 7.2, 0, 0, 0}},
                                  {"staged64x128", 64, 128, 3, {0.32, 0.39, 6.0, 0.074, 0, 0}, {0.40, 0.30, 5.9, 0, 0, 0}},
                                  {"staged64x64", 64, 64, 4, {0.228, 0.2725, 4.5, 0.046, 2.4, 2.1e-6}, {0.165, 0.238, 4.3, 0, 2.7, 1.9e-6}}};

inline GemmChoice choose_gemm(const GemmShape& s, int cus, uint64_t partial_bytes) {
  GemmChoice c;
  if (strcmp(s.dtype, "f32") == 0) {
    double us = 1e30;
    for (const F32Strip& r : kF32Strips) {
      const F32Plan p = f32_plan(r, s.m, s.n, s.k, cus, partial_bytes);
      if (s.y_cols >= 64 && p.us < us * 0.98) us = p.us, c.strip = &r, c.strip_plan = p;
    }
    if (c.strip) snprintf(c.variant, sizeof(c.variant), "f32_%s", c.strip->kernel);
    c.needs_room = c.strip && c.strip_plan.splits > 1;
    return c;
  }
  if (s.k <= 64) return c;   // one K tile: nothing to stage, split or overlap
  auto pick = [&](const char* kernel) { snprintf(c.variant, sizeof(c.variant), "%s_%s", s.dtype, kernel); };
  // Few rows.  Measured at 1 to 64 rows, f16 and bf16 (us, thin against 128 x 128 tiles): 4096 x 4096 10 - 21 against 53,
  // K = 14336 25 - 41 against 175, 14336 x 4096 24 - 35 against 54, 1024 x 1024 5 - 9 against 11.  128-column strips where
  // there are enough of them to keep three quarters of the compute units busy (28672 x 8192, one row: 83 us against 92).
  // With more than 32 rows a workgroup fills a compute unit by itself (139 KB of partial sums), so strips are the better ones only while
  // they fit the chip once: over 459 products of 33 to 64 rows the tiles chosen below take 0.55 to 0.98 times the strips' time beyond 16384
  // columns, 0.76 in the mean (us: 60 x 19072 x 448 12.5 against 9.0 and 7.5 from memory and from the caches), and the best of them 1.10 up to there.
  // Up to 128 rows (two passes over y, the second from L2) while the strips of both passes fit the chip once
  // (4096 x 4096 23 us against 27 with staged tiles; 14336 x 4096 60 against 46).
  // From 96 strips of 128 columns on where y is streamed past the caches (4096 x 14336, 112 strips and two workgroups to each: 22.1 us, 64-column strips 23.0).
  const bool many = s.n >= 192 * 128 || (s.m <= 16 && s.n >= 96 * 128 && streamed_past_caches(s.n, s.k));
  const int64_t strips = (s.n + 63) / 64;
  // 128 x 128 tiles whose K is shared read y once for all the rows, in as many workgroups: from 49 rows on they are the better ones where K is
  // long enough to be shared (f16, us on strips and on tiles: 112 x 3584 x 10496 43.6, 30; 64 x 2240 x 7680 28.7, 19; 97 x 576 x 3968 18.6, 13.6;
  // below that line 53 x 3648 x 1984 13.0, 12.9; 120 x 4032 x 1280 10.7, 11.3), and where there is room for more than two workgroups to a
  // tile or K is very long (58 x 13376 x 4096 29.7, 30.1; 56 x 14784 x 16256 104, 88).  Of up to 48 rows a strip multiplies three
  // quarters of what it does of 64, and the two are near each other (47 x 3968 x 12096 30.2, 27.9; 39 x 8256 x 2816 18.2, 17.1; 35 x 15936 x
  // 3328 23.8, 30.4), and one or two tiles of at most 64 rows stay on strips too.  Over 180 products beyond the line 0.70 of the strips' time.
  const uint64_t wide = tiles_of(s.m, s.n, 128, 128);
  const bool tiles_share = s.aligned && strcmp(s.dtype, "bf16f32") != 0 && partial_bytes > 0 && s.m > 48 && (s.m > 64 || wide > 2) && s.k >= 28 * 64 &&
                           (wide * 8 <= (uint64_t)cus * 3 || s.k >= 96 * 64);
  if (s.y_cols >= 64 && !tiles_share && (s.m <= 32 || (s.m <= 64 && strips <= cus) || (s.m <= 128 && 2 * strips <= cus))) {
    pick(s.m > 32 ? "thin64x64" : s.m > 16 ? "thin32x64" : many && s.y_cols >= 128 ? "thin16x128" : "thin16x64");
    return c;
  }
  auto tiles = [&](int bm, int bn) { return (uint64_t)((s.m + bm - 1) / bm) * (uint64_t)((s.n + bn - 1) / bn); };
  const double kt = s.k / 64.0;
  double best = 1e30;
  const char* picked = nullptr;
  bool shares_k = false;   // the kernel picked
  // (up to K = 512 the start and the output of a tile are most of a launch: the partition's own tile, if it has kernels)
  const bool ring = s.aligned && (s.k > 512 || !s.own_tile) && strcmp(s.dtype, "bf16f32") != 0;
  if (ring)
    for (const RingTile& r : kRingTiles) {
      // a handful of tiles of a short K: 64 x 64 staged ones, priced below (us there and on 128 x 128: 263 x 64 x 1728 9.4, 10.8; 141 x
      // 320 x 2496 11.3, 12.3; beyond, 250 x 384 x 4352 16.3, 14.4)
      if (s.k <= 2560 && tiles_of(s.m, s.n, 128, 128) < 16) break;
      const RingPlan p = cutile::ring_plan(r, s.m, s.n, s.k, cus, partial_bytes, s.whole_k);
      // (128 x 256 against 256 x 128, f16: 619 x 8832 x 4096 56.7 us, 59.0; 620 x 5000 x 4096 40.8, 39.6; 600 x 8192 x 4096 54.1, 55.8; equal for
      // bf16: the prices are good to 5 %, so only where it is the cheaper one by more)
      if (p.us < best * (r.bm < r.bn && r.bm == 128 ? 0.94 : 0.98)) best = p.us, picked = r.kernel, shares_k = p.splits > 1, c.ring = &r, c.ring_plan = p;
    }
  // Staged tiles: the only ones for unaligned rows (6198 x 3583 x 1194 f16 1150 -> 86 us, 200 x 50021 x 1024 bf16 587 -> 37 us), and,
  // split along K, the better ones for outputs of less than about 64 tiles of 128 x 128.
  // (of more tiles, aligned and of a partition without kernels of its own, ring tiles are the better ones for any K: 105 products of 128 tiles and more, with staged
  // ones 1.01 to 1.17 times the best one's time by their K, 2966 x 9808 x 2832 224 us, ring 154)
  if (ring ? tiles(128, 128) < (uint64_t)cus / 2 : !s.own_tile) {
    // 256 x 256 has the fewest bytes per product and pays most for start and output (bf16, us on it and on the best other: 200 x 50021 x 1024 37.3, 46.3;
    // 1000 x 20001 x 1024 67, 62; 961 x 7277 x 2155 57, 44), with a short K in many rounds most of all (5587 x 30444 x 164 240, 181 on 64 x 128: nothing
    // runs beside a start or an output on the tiles that fill a compute unit by themselves).  Of aligned rows 64 x 64 tiles that share K are the better ones of few outputs (us there and on the
    // ring: 1919 x 64 x 3264 10.9, 13.9; 173 x 832 x 3328 11.5, 14.2; 100 x 1024 x 4096 11.8, 14.3), and without a workspace of more (309 x 2240 x 5184 25, 31; 150 x
    // 3456 x 9536 57, 81): over those 520 products, and over 680 more of sizes that models have, the kernel priced
    // lowest takes 1.004 of the best one's time (1.02 before, 1.16 without a workspace).
    for (const StagedTile& r : kStaged) {
      if (s.y_cols < r.bn || (ring && r.bm == 256)) continue;
      const uint64_t t = tiles(r.bm, r.bn), sk = partial_bytes ? staged_splits(r.bm, r.bn, t, s.k, cus) : 1;
      const uint64_t slots = (uint64_t)cus * r.per_cu, rounds = t * sk / slots, rest = t * sk % slots;
      if (r.per_cu == 1 && rounds >= 2 && kt < 8) continue;
      const StagedTile::Prices& a = ring ? r.aligned : r.any;
      const double ends = a.ends + (r.bn == 256 && s.k % 64 != 0 ? 1.8 : 0.0);   // (there a ragged K tile stands behind the sequence)
      auto round = [&](uint64_t each) { return kt / (double)sk * std::max(a.one, a.more * (double)each) + ends; };
      double us = ((double)rounds * round(r.per_cu) + (rest ? round((rest + cus - 1) / cus) : 0.0)) * (s.x_aligned ? 1.0 : 1.0 + a.x) +
                  (sk > 1 ? a.split + a.sum * (double)(s.m * s.n * (int64_t)sk) : 0.0);
      // (a row of tiles of a large y: at 3.5 TB/s, ring tiles have more of it in flight; us here and there 54 x 7680 x 6272 34.3, 29.2; 64 x 4096 x 4096 18.0, 14.8)
      if (ring && s.m <= 64) us = std::max(us, a.ends + a.split + (double)(s.n * s.k) * 2 / 3.5e6);
      if (ring && r.bm == 64 && r.bn == 64 && partial_bytes && t <= 2 * (uint64_t)cus && s.m > 64) {
        const StagedPlan p = staged_plan(s.m, s.n, s.k, cus);
        if (us < best * 0.98 || p.us < best * 0.96) picked = r.kernel, shares_k = p.splits > 1, c.ring = nullptr, c.staged = p.splits;
        continue;
      }
      if (us < best * (ring ? 0.98 : 1.0)) best = us, picked = r.kernel, shares_k = sk > 1, c.ring = nullptr;
    }
  }
  if (picked) pick(picked);
  c.needs_room = shares_k || tiles_share;   // (strips that were passed over share K inside a workgroup, and need none)
  return c;
}

// ---- block-scaled products ----
struct ScaledShape {
  int64_t m, n;
  int32_t pieces;          // 64-byte pieces of a row: 64 (fp8) or 128 (fp4) values of K
  bool fp4;
};
// K splits of a scaled_flat.hip launch: up to half the compute units busy, at least two 128-byte steps for each of the 8
// wavefronts (mxfp8, 64 x 1024 x 8192, 32 strips: 16.7, 13.2, 12.5 us with 1, 2, 4 splits; 16 x 4096 x 4096, 64 strips: 9.4,
// 9.4, 10.5; nvfp4 of that size 9.9, 11.7, 13.1; 16 x 1024 x 1024 6.6, 8.0, 8.5).
inline uint32_t scaled_splits(uint64_t blocks, int32_t pieces, int cus) {
  return (uint32_t)std::max<int64_t>(1, std::min<int64_t>((int64_t)((uint64_t)cus / 2 / std::max<uint64_t>(blocks, 1)), pieces / (2 * 8 * 2)));
}
// As launched, which the prices below do not know: strips of up to 64 x 64 outputs, whose partial sums are few, in one round of a workgroup to each compute unit, and
// finer where K is long (partial sums are read eight at a time, split_k.h).  Operands from memory, us as above and so: mxfp8 8 x 4096 x 4096 10.0, 9.3; 1 x 5120 x
// 5120 15.5, 11.1; 60 x 4096 x 4096 14.2, 12.5; 8 x 896 x 5248 9.3, 7.4; nvfp4 1 x 1088 x 6656 13.2, 10.4; 8 x 896 x 5248 13.4, 10.6.  (Shorter ones in
// two instead of one: mxfp8 16 x 2048 x 2048 6.5, 7.7; nvfp4 8 x 4096 x 4096 9.4, 10.8; and mxfp8 of less than 90 pieces and up to 32 rows where strips leave room for two only:
// 15 x 8128 x 4736 11.1, 12.4; 1 x 8000 x 4096 9.1, 9.9; 12 x 7424 x 5632 12.2, 13.0; beyond, 2 x 8192 x 7552 20.2, 16.1.)  Over 110 products that are
// shared finer than priced, of 1 to 100 rows, 0.85 of the time as priced, the slowest 1.02.
inline uint32_t scaled_launch_splits(uint64_t blocks, int32_t pieces, int cus, bool fp4, int bm, int bn) {
  const uint32_t priced = scaled_splits(blocks, pieces, cus);
  if (bm * bn > 64 * 64) return priced;
  const int64_t fit = (int64_t)((uint64_t)cus / std::max<uint64_t>(blocks, 1));
  const int64_t most = fp4 ? pieces / 20 : pieces < 64 ? pieces / 32 : fit == 2 && bm < 64 && pieces < 90 ? 1 : pieces / 16;
  return std::max(priced, (uint32_t)std::max<int64_t>(1, std::min<int64_t>({fit, most, 8})));
}
// fp8 on 128 x 128 tiles that have a compute unit each (mxfp8_tiles.hip), K shared by up to 8 workgroups in whole blocks of 512 positions: us a K tile
// of 128 where few compute units are busy and where all are, us of start and output, and of partial tiles (113 times of 54 products, 9.5 % rms).
// Against the two-stage kernel: 1000 x 4096 x 4096 26.5 -> 22.3 us, 1943 x 1472 x 7296 50 -> 37, 459 x 4416 x 512 7.6 -> 6.6; against strips, with K
// shared by two: 859 x 1600 x 5888 28.4 -> 19.6, 360 x 4352 x 6912 35 -> 28.
struct MxPlan {
  uint32_t splits;   // 0: more tiles than compute units
  double us;
};
inline MxPlan mx_plan(int64_t m, int64_t n, int32_t pieces, int cus, uint64_t partial_bytes) {
  const uint64_t t = tiles_of(m, n, 128, 128);
  const int64_t kt = pieces / 2;
  MxPlan best{0, 1e30};
  for (uint32_t s : {1u, 2u, 3u, 4u, 6u, 8u}) {
    const uint64_t g = t * s;
    if (g > (uint64_t)cus || (s > 1 && (kt < 8 * s || g * 128 * 128 * 4 > partial_bytes))) break;
    const double tiles = s > 1 ? (double)((kt + 4 * s - 1) / (4 * s) * 4) : (double)kt;
    const double us = tiles * (0.405 + 0.255 * (double)g / cus) + 4.3 + (s > 1 ? (4.4e-5 * s + 1e-6 * (double)g) * 128 * 128 : 0.0);
    if (us < best.us * 0.98) best = {s, us};
  }
  return best;
}
// Strips of scaled_flat.hip, us a piece of K of each format while they fit the chip once; and of fp4 strips in more rounds than one, a piece in a round that
// few and that all compute units have, and start and output of a round.
struct FlatStrip {
  const char* name;
  int bm, bn;
  double fp8, fp4, few, all, ends;
};
constexpr FlatStrip kFlat[] = {{"flat16x64", 16, 64, 0.09, 0.20, 0.20, 0.20, 5.5}, {"flat32x64", 32, 64, 0.12, 0.28, 0.28, 0.28, 5.5}, {"flat64x64", 64, 64, 0.155, 0.36, 0.294, 0.297, 4.5},
                               {"flat64x128", 64, 128, 0.27, 0.62, 0.534, 0.561, 4.8}, {"flat128x128", 128, 128, 0.52, 1.12, 1.053, 1.08, 5.4}};
// The kernel by name, or nullptr: the partition's own (tuning record, then the table's order).  us per 64-byte piece of K for
// one block on each compute unit, measured at K = 4096 (mxfp8: 16 x 4096 9.4 us, 64 x 4096 13.4, 512 x 4096 21 on 64 x 128 blocks, 24 with
// 128 x 128 tiles; nvfp4: 9.9, 14.7, 24).  The 256 x 256 kernels are the better ones where their tiles come near to filling the chip.
// `lone`: what mx_plan says for fp8, where it was asked.
inline const char* choose_scaled(const ScaledShape& s, int own_m, int own_n, int cus, uint64_t partial_bytes, MxPlan* lone) {
  // a partition whose output other tiles of nvfp4_gemm.hip may compute too
  const bool tiled = s.fp4 && own_m == own_n && (own_m == 128 || (own_m == 256 && s.pieces > 4));
  auto blocks = [&](int bm, int bn) { return (uint64_t)((s.m + bm - 1) / bm) * (uint64_t)((s.n + bn - 1) / bn); };
  // fp4 of up to 128 values: too short for strips; start and output of a 256 x 256 tile are most of it (us there and on 128 x 128: 256 x 128
  // 9.2, 5.5; 988 x 5056 14.8, 9.7; 381 x 15296 15.0, 10.4; of more than a round of the small ones 1504 x 10432 16.3, 18.4)
  if (s.fp4 && s.pieces <= 1) return own_m == 256 && own_n == 256 && blocks(128, 128) <= 2 * (uint64_t)cus ? "128x128x64_w2x2" : nullptr;
  if (s.pieces <= 4 && !tiled) return nullptr;   // two steps: nothing to share out
  if (!tiled && s.m > 64 && own_m == 256 && own_n == 256 && blocks(256, 256) * 4 >= (uint64_t)cus * 3) return nullptr;
  // (fp8 on 128 x 128: the direct pipeline below is always the cheaper one; only a name reaches flat128x128 there)
  const char* name = nullptr;
  double best = 1e30;
  auto rounds = [&](uint64_t g, uint64_t at_once, double few, double all, double ends) {
    const uint64_t rest = g % at_once;
    return (double)(g / at_once) * (all * s.pieces + ends) + (rest ? (few + (all - few) * (double)rest / (double)at_once) * s.pieces + ends : 0.0);
  };
  for (const FlatStrip& k : kFlat) {
    const uint64_t b = blocks(k.bm, k.bn), waves = (b + cus - 1) / cus;
    if (s.pieces <= 4) break;
    const double us = s.fp4 && waves > 1 ? rounds(b, cus, k.few, k.all, k.ends) : (double)waves * ((s.fp4 ? k.fp4 : k.fp8) * s.pieces / scaled_splits(b, s.pieces, cus) + 3.5);
    if (us < best) best = us, name = k.name;
  }
  if (tiled) {
    // Whole tiles, expanded to f16 once for the workgroup: 256 x 256 to a compute unit, or two of 128 x 128 (2.37 a piece as soon as any has two).  Least
    // squares, as for strips in several rounds, over 400 products of 17 to 4096 rows, operands from memory, every kernel timed (256 x 256 2.6 % rms, 128 x 128 7.8, strips 5):
    // the kernel priced lowest takes 1.035 of the best one's time, and nowhere more than 1.04 of what strips and two-stage tiles alone took, where prices
    // by rounds of strips and a tile's own had taken up to 1.24 (bf16 out, us on 256 x 256, 128 x 128 and the best strips: 2476 x 6080 x 896 34.7, 44.7, 54.7;
    // 2940 x 5568 x 1152, 264 of the large tiles, 75, 54, 60; 4096 x 4096 x 4096 117, 162, 153; 1024 x 4096 x 4096 101, 53, 44; 1587 x 3328 x 7040 176, 124, 107).
    const uint64_t small = blocks(128, 128), rest = small % (2 * (uint64_t)cus);
    const double us256 = rounds(blocks(256, 256), cus, 2.48, 3.42, 12.1);
    const double us128 = (double)(small / (2 * (uint64_t)cus)) * (2.48 * s.pieces + 4.5) +
                         (rest <= (uint64_t)cus ? rounds(rest, cus, 0.87, 1.62, 4.5) : (2.37 + 0.11 * (double)(rest - cus) / cus) * s.pieces + 4.5);
    if (us128 < best) best = us128, name = "128x128x64_w2x2";
    if (us256 < best) best = us256, name = "256x256x64_q2x4";
    return name;
  }
  if (!s.fp4) {
    *lone = mx_plan(s.m, s.n, s.pieces, cus, partial_bytes);
    if (lone->splits && lone->us < best) best = lone->us, name = "128x128x128_e2x2";
  }
  if (!s.fp4 && blocks(128, 128) > (uint64_t)cus) {   // two workgroups to a compute unit
    const uint64_t b = blocks(128, 128), rest = b % (2 * (uint64_t)cus);
    const double us = (double)(b / (2 * (uint64_t)cus)) * (0.58 * s.pieces + 4) + (rest == 0 ? 0.0 : (rest <= (uint64_t)cus ? 0.31 : 0.58) * s.pieces + 4);
    if (us < best) best = us, name = "128x128x128_e2x2";
  } else if (own_m == 256 && own_n == 256) {
    const uint64_t b = blocks(256, 256), waves = (b + cus - 1) / cus;
    const double part = (double)std::min<uint64_t>(b, cus) / cus;
    const double us = (double)waves * (s.pieces * (1.85 + 2.1 * std::max(0.0, part - 0.25) / 0.75) + 4);
    if (us < best) return nullptr;
  }
  return name;
}

}  // namespace cutile
