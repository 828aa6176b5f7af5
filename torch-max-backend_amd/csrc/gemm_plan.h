// Host-side choices of the GEMM family that do not depend on the storage type's kernels: which
// operands the matrix-core kernels take, and when a product is split along K.
#pragma once

#include <cmath>

#include "gemm_mfma.h"
#include "gemm_f32_wide.h"

namespace tmb {

static inline bool mfma_eligible(const GemmArgs& g, int64_t batch, int trans_a, int trans_b) {
  if (trans_a) return false;
  if (g.k % 8 != 0 || g.lda % 8 != 0 || g.ldb % 8 != 0) return false;
  if (!aligned16(g.a) || !aligned16(g.b)) return false;
  if (batch > 1 && (g.stride_a % 8 != 0 || g.stride_b % 8 != 0)) return false;
  if (g.m < 1 || g.n < 1 || g.k < 8) return false;
  // the kernel addresses operands with 32-bit byte offsets from their base
  const int64_t a_span = g.m * g.lda * 2, b_span = (trans_b ? g.n : g.k) * g.ldb * 2;
  if (a_span >= (int64_t{1} << 32) || b_span >= (int64_t{1} << 32)) return false;
  (void)trans_b;
  return true;
}

// A stored [K, M] with B stored [K, N] (the weight-gradient product) on the ring kernels: whole 16-byte
// chunks along m and n, whole stages of K and enough of them for the ring.
static inline bool mfma_transposed_a_eligible(const GemmArgs& g, int64_t batch, int trans_a, int trans_b,
                                              int epilogue) {
  if (!trans_a || trans_b || epilogue != TMB_EPI_NONE) return false;
  if (g.k % 32 != 0 || g.k < 256 || g.m % 8 != 0 || g.n % 8 != 0 || g.n <= 64) return false;
  if (g.lda % 8 != 0 || g.ldb % 8 != 0 || !aligned16(g.a) || !aligned16(g.b)) return false;
  if (batch > 1 && (g.stride_a % 8 != 0 || g.stride_b % 8 != 0)) return false;
  const int64_t a_span = g.k * g.lda * 2, b_span = g.k * g.ldb * 2;
  return a_span < (int64_t{1} << 32) && b_span < (int64_t{1} << 32);
}

// Shapes the stream kernel takes: K = 64, whole 128 x 128 tiles, 16-byte aligned operands whose
// rows are whole 16-byte chunks, no epilogue beyond the bias, no residual.
static inline bool stream64_eligible(const GemmArgs& g, int64_t batch, int trans_b, int epilogue) {
  if (g.k != 64 || g.m % 128 != 0 || g.n % 128 != 0 || epilogue != TMB_EPI_NONE) return false;
  if (g.residual != nullptr || g.out_f32) return false;
  if (g.lda % 8 != 0 || g.ldb % 8 != 0 || !aligned16(g.a) || !aligned16(g.b)) return false;
  if (batch > 1 && (g.stride_a % 8 != 0 || g.stride_b % 8 != 0)) return false;
  // lane offsets are 32-bit byte offsets inside one tile's rows
  const int64_t a_span = 128 * g.lda * 2, b_span = (trans_b ? 128 : 64) * g.ldb * 2;
  if (a_span >= (int64_t{1} << 32) || b_span >= (int64_t{1} << 32)) return false;
  const int64_t tiles = (g.m / 128) * (g.n / 128) * batch;
  return tiles >= 512 && tiles < (int64_t{1} << 40);
}

// Tiles of the kernel for products that leave most of the chip idle (gemm_small.h), and what a
// launch with one of them takes, in microseconds: a start, then per tile its operands' bytes at the
// rate one workgroup's loads sustain and the way of its partial tiles through LDS. A CU that gets a
// second workgroup of the tiles that fit it twice (up to 32 x 32) loads faster than one alone,
// hence the power; the two large ones take a CU's LDS and run in whole rounds. The constants are a
// fit to 720 shapes (1 .. 2048 rows, 256 .. 8192 columns, K 64 .. 4096, both layouts of B), within
// 15 % of them.
struct SmallTile {
  int bm, bn, waves;
  double start, bytes_per_us, lds;
  bool alone;
};
constexpr SmallTile kSmallTiles[] = {{16, 16, 8, 2.8, 60e3, 0.4, false}, {16, 32, 8, 2.8, 70e3, 0.7, false},
                                     {32, 32, 8, 2.8, 80e3, 1.0, false}, {32, 32, 4, 3.0, 70e3, 0.4, false},
                                     {32, 64, 8, 2.8, 90e3, 1.5, true},  {64, 64, 8, 3.0, 90e3, 2.0, true}};
constexpr int kSmallTileCount = sizeof(kSmallTiles) / sizeof(kSmallTiles[0]);

static inline int small_tile(int64_t batch, int64_t m, int64_t n, int64_t k) {
  int best = 0;
  double least = 0.0;
  for (int i = 0; i < kSmallTileCount; ++i) {
    const SmallTile& t = kSmallTiles[i];
    const int64_t tiles = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * batch;
    double rounds = 1.0;
    if (tiles > 256) rounds = t.alone ? static_cast<double>((tiles + 255) / 256) : std::pow(tiles / 256.0, 0.9);
    const double cost = t.start + rounds * ((t.bm + t.bn) * 2.0 * k / t.bytes_per_us + t.lds);
    if (i == 0 || cost < least) {
      least = cost;
      best = i;
    }
  }
  return best;
}

// Which products that kernel takes (16-bit operands, A row-major): those whose 64 x 64 tiles fit one
// round of the 256 CUs, up to K = 4096 (at K = 8192 the split-K launch is level with it), and 16 rows
// or fewer against any number of columns, which is a pass over B. Measured over the 600 such shapes
// of the sweep above it is 1.8 times as fast as what ran before (128 x 768 x 768 8.9 -> 3.6 us,
// 32 x 2304 x 768 11.5 -> 4.0, 128 x 768 x 3072 13.4 -> 6.2, 1024 x 768 x 3072 19.9 -> 14.3 us; two
// N-major shapes of 600 run 5-10 % longer), and over what lies outside on average slower.
static inline bool small_applies(int64_t batch, int64_t m, int64_t n, int64_t k) {
  // (64 columns or fewer are not split, and 256 x 64 tiles leave most of the chip idle: 300 x 64 x 8192 155 -> 15 us,
  // 3264 x 48 x 6720, N-major, 482 -> 22)
  if ((k > 4096 && n > 64) || k > 16384 || k < 8 || m < 1 || n < 1) return false;
  if (m <= 16 && batch == 1) return true;
  return ((m + 63) / 64) * ((n + 63) / 64) * batch <= 256;
}
int gemm_small(const GemmArgs& g, int64_t batch, int tile, int trans_b, bool bf16, int epilogue, hipStream_t stream);

// 16-bit operands in any layout and at any alignment (gemm_any.h): tile and split count. A launch takes,
// in microseconds, a start and per round of tiles their operands' bytes at the rate a workgroup's
// unaligned pieces arrive (half of the aligned kernel's above) and the partial tiles' way through LDS;
// several workgroups share a CU, hence the power instead of whole rounds. Fitted to 70 shapes of 8 .. 8192
// rows, 64 .. 50257 columns and K 64 .. 30001 in all layouts, within 15-20 % (rms) of each tile; the tile
// it picks takes 3 % longer than the best one on average. A split adds its reduction.
struct AnyTile {
  int bm, bn;
  double start, bytes_per_us, lds, power;
};
constexpr AnyTile kAnyTiles[] = {{16, 16, 3.4, 38e3, 0.3, 1.08}, {16, 32, 3.1, 44e3, 0.9, 1.0},
                                 {32, 32, 3.1, 49e3, 1.0, 1.02}, {32, 32, 3.5, 41e3, 0.5, 0.96},
                                 {64, 64, 2.6, 43e3, 3.7, 0.88}};
struct AnyPlan {
  int tile;    // index into kAnyTiles
  int splits;  // 0: not split
  double cost;
};
static inline AnyPlan any_plan(int64_t batch, int64_t m, int64_t n, int64_t k, bool may_split) {
  AnyPlan p{0, 0, 0.0};
  auto consider = [&](int splits) {
    const int64_t runs = splits > 0 ? splits : batch;
    const double depth = static_cast<double>(k) / (splits > 0 ? splits : 1);
    for (int i = 0; i < static_cast<int>(sizeof(kAnyTiles) / sizeof(kAnyTiles[0])); ++i) {
      const AnyTile& t = kAnyTiles[i];
      const double tiles = static_cast<double>((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * runs;
      const double rounds = tiles <= 256.0 ? 1.0 : std::pow(tiles / 256.0, t.power);
      double cost = t.start + rounds * ((t.bm + t.bn) * 2.0 * depth / t.bytes_per_us + t.lds);
      if (splits > 0) cost += 5.5 + 1e-6 * splits * m * n;
      if (p.cost == 0.0 || cost < p.cost) p = AnyPlan{i, splits, cost};
    }
  };
  consider(0);
  if (may_split && batch == 1 && m * n < (int64_t{1} << 31))
    for (const int s : {2, 3, 4, 6, 8, 12, 16})
      if (k >= 192 * s) consider(s);
  return p;
}
// Short K over many tiles, against the vector kernel: the waves of a workgroup share 64-deep slices (32-deep in
// fp32), so with one slice or less all but one of them idle, and a launch of many tiles takes what a tile's
// way through LDS takes. The vector kernel's 64 x 64 tiles are then faster (bf16 7309 x 3268 x 2 31 against 70 us, 48 x
// 402 x 354 x 8 14 against 26; fp32 48 x 5222 x 7 x 5 17 against 55). Microseconds of both, a start and rounds of tiles,
// fitted to 1200 unaligned shapes a type of 2 .. 9000 in each extent, half of them K <= 128, 1 .. 48 batches; 12-17 %
// (rms; a wave-sharing tile's power law 15-20 % in 16 bits). By the times measured on those shapes with each kernel
// forced, 97 of 1200 (fp32 287) would take a tenth longer than on the vector kernel or on padded copies if the waves'
// kernels took them all, and 4 (16) do with the rules here.
struct ManyTiles {
  double start, per_k, per_tile, power;
};
constexpr ManyTiles kAnyMany[] = {{3.1, 0.00157, 0.585, 0.991}, {2.9, 0.00204, 1.11, 0.986}, {3.2, 0.00262, 1.355, 0.978},
                                  {3.8, 0.00285, 0.637, 0.972}, {2.9, 0.00604, 3.21, 0.919}};
static inline double many_tiles_cost(const ManyTiles& t, int bm, int bn, int64_t batch, int64_t m, int64_t n, int64_t k) {
  const double r = static_cast<double>(((m + bm - 1) / bm) * ((n + bn - 1) / bn)) * batch / 256.0;
  return t.start + (r <= 1.0 ? 1.0 : std::pow(r, t.power)) * (t.per_k * k + t.per_tile);
}
static inline double simt_cost(bool f32, int64_t batch, int64_t m, int64_t n, int64_t k) {
  const double tiles = static_cast<double>(((m + 63) / 64) * ((n + 63) / 64)) * batch, r = tiles / 256.0;
  const double filled = static_cast<double>(m) * n * batch / (tiles * 4096.0);
  const double alone = f32 ? 0.15 * k - 0.7 : 0.15 * k - 0.5;
  const double many = f32 ? r * (0.030 * k + 0.31 + 1.21 * filled) : r * (0.036 * k + 0.21 + 0.72 * filled);
  return (f32 ? 4.8 : 5.1) + (alone > many ? alone : many);
}
static inline bool simt_instead_of_any(const GemmArgs& g, int64_t batch, const AnyPlan& plan) {
  if (g.residual != nullptr || plan.splits > 0 || g.k > 32) return false;
  const AnyTile& t = kAnyTiles[plan.tile];
  return simt_cost(false, batch, g.m, g.n, g.k) <
         many_tiles_cost(kAnyMany[plan.tile], t.bm, t.bn, batch, g.m, g.n, g.k);
}
// What that kernel asks of its operands: eight elements along each contiguous direction, and lane
// offsets within a tile that fit 32 bits.
static inline bool any_eligible(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int trans_a, int trans_b) {
  if (m < 1 || n < 1 || k < 1) return false;
  if ((trans_a ? m : k) < 8 || (trans_b ? k : n) < 8) return false;
  return lda < (int64_t{1} << 23) && ldb < (int64_t{1} << 23);
}
// Products whose 256 x 128 tiles leave CUs idle (K a multiple of 64, four stages or more): the largest tile that still
// runs in one round, one workgroup of eight waves to a CU (64-deep stages, three or four in LDS), of 64 x 128 (A row-major
// only: a 64-wide A stored [K, M] has too few 16-byte chunks a row for its swizzle) and 128 x 128. What bounds them is the
// wait for a stage, which two waves a SIMD cover and four did not: bf16, the 128 x 128 x 32 tiles of four waves
// that ran before against these, microseconds: 2100 x 768 x 768 11.9 and 8.2, 3400 x 768 x 768 12.1 and 10.2, 2700 x
// 768 x 3072 33.5 (split) and 24.5, dy^T x 3072 x 768 x 2048 27.5 (split) and 19.3. Beyond one round 64 x 128 tiles,
// two workgroups to a CU, of three stages: 5400 x 768 x 768 17.5 and 12.1, 5400 x 768 x 3072 50.4 and 42.8.
enum { kRing64x128 = 1, kRing128x128 = 2 };
static inline int ring_one_round(int64_t batch, int64_t m, int64_t n, int64_t k, int trans_a) {
  if (k % 64 != 0 || k < 256) return 0;
  const int64_t tiles_n = (n + 127) / 128 * batch;
  if (!trans_a && (m + 63) / 64 * tiles_n <= 256) return kRing64x128;
  return (m + 127) / 128 * tiles_n <= 256 ? kRing128x128 : 0;
}
// Their microseconds, within 10 % at K 512 .. 4096 (the more of the chip is busy, the slower it runs).
static inline double one_round_cost(int form, int64_t t128, int64_t k) {
  if (form == kRing64x128) return 4.1 + 0.0043 * k;
  return 5.2 + k * (0.0060 + 0.0030 * std::fmin(std::fmax((t128 - 128) / 96.0, 0.0), 1.0));
}
// The same 128 x 128 form for the runs of a split product that has a CU for each: 6 .. 11 % faster than the four waves'
// (dy^T x 1408 x 832 x 6144 30.2 and 27.5 us, 2304 x 768 x 4096 30.4 and 27.3), except where the chip is full and the runs
// are short (1700 x 768 x 3072 in three 22.3 and 24.9).
static inline bool splitk_eight_waves(int64_t t128, int64_t k, int splits) {
  const int64_t units = t128 * splits;
  return k % 64 == 0 && units <= 256 && (units <= 232 || k >= 1152 * splits);
}

// Microseconds of a product on the ring kernels: 900 TFLOP/s in rounds of 128 x 128 tiles, two per CU.
static inline double ring_cost(int64_t batch, int64_t m, int64_t n, int64_t k) {
  const double tiles = static_cast<double>((m + 127) / 128) * ((n + 127) / 128) * batch;
  return 6.0 + (tiles <= 256.0 ? 0.011 * k : std::ceil(tiles / 512.0) * 0.0186 * k);
}
// Microseconds of the other way for the same operands: copy what the ring kernels cannot read into padded buffers (3 us and
// the bytes at 4 TB/s each), then multiply there. A transposing copy counts as one at 1 TB/s: it runs at four, but counted
// so products go that way whose launches then take longer (64 x 5298 x 512 with its backward 54 us for 32). Within 15 % of
// the measured sum for products from 10 GFLOP on (4099^3 198 against 197, 4383 x 1568 x 1228 38 against 38, 1829 x 3429 x
// 4716 147 against 156).
struct SplitKPlan {
  int splits;  // 0: not used
  int tile;    // 128 or 256
  double cost;
};
static inline SplitKPlan splitk_or_whole(int64_t batch, int64_t m, int64_t n, int64_t k, int trans_a);
static inline double padded_cost(int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, bool a_ok,
                                 bool b_ok, int trans_a, int trans_b, bool plain) {
  double cost = ring_cost(batch, m, n, k);
  const int64_t depth = k % 8 == 0 ? k : (k + 63) / 64 * 64;
  const SplitKPlan split = splitk_or_whole(batch, m, n, depth, trans_a);
  if (split.splits > 0 && (trans_a || !small_applies(batch, m, n, depth)))
    cost = std::fmin(cost, split.cost + 6.0);  // (2336 x 512 x 8672 57 us so, 81 where it lies)
  else if (const int form = ring_one_round(batch, m, n, depth, trans_a); form != 0 && k >= 2048)
    cost = one_round_cost(form, ((m + 127) / 128) * ((n + 127) / 128) * batch, depth);
  auto copy = [&](int64_t elements, bool transposing) {
    return 3.0 + static_cast<double>(elements) * batch * 4.0 / (transposing ? 1e6 : 4e6);
  };
  const bool b_fits = b_ok && ldb % 8 == 0;
  if (trans_a) {
    const bool keeps_form = plain && batch == 1 && b_fits && !trans_b && k % 32 == 0 && k >= 256 && n % 8 == 0 && n > 64;
    if (keeps_form) return cost + copy(m * k, false);
    cost += copy(m * k, true) + (k % 8 != 0 ? copy(m * k, false) : 0.0);
  } else if (k % 8 != 0 || lda % 8 != 0 || !a_ok) {
    cost += copy(m * k, false);
  }
  if (trans_b ? !b_fits || k % 8 != 0 : b_fits && k % 8 != 0) cost += copy(n * k, false);
  else if (!trans_b && !b_fits) cost += copy(n * k, true);
  return cost;
}
int gemm_any(const GemmArgs& g, int64_t batch, int tile, int trans_a, int trans_b, bool bf16, int epilogue,
             hipStream_t stream);

// A transposed A with a residual that the rings would multiply without one and that is rounded with the product once:
// whether the any-layout kernel, which takes the residual along, is faster than their product and the caller's four
// launches in float32 (5.8 TB/s). 4096^3: 241 us there against 193 apart, 768 x 3072 x 1024 24 against 31, 2048^3 40
// against 46, 1024^3 14 against 27, 8192 x 8192 x 1024 420 against 492. The fifth is the models' own error.
static inline bool any_with_residual_pays(const GemmArgs& g, int64_t batch, double any_cost) {
  const double add = 12.0 + static_cast<double>(g.m) * g.n * batch * 30.0 / 5.8e6;
  return any_cost * 1.2 < ring_cost(batch, g.m, g.n, g.k) + add;
}

// Split-K: products with few output tiles and a long K (weight gradients, narrow projections)
// leave most CUs idle. K is cut into `splits` runs of whole stages (equal to within one stage)
// that run as the y dimension of one launch of a ring kernel and store fp32 partials
// [splits][M][N] into a workspace; a second kernel adds them in split order and applies bias,
// epilogue and the one cast, so the result is still "fp32 accumulation, one rounding" and depends
// on the shape only.
//
// Tile and split count come from a small cost model (all in microseconds): the 256 x 256 x 64
// kernel sustains about 1240 TFLOP/s over 256 one-per-CU workgroups, the 128 x 128 x 32 kernel
// about 900 TFLOP/s over 512 two-per-CU workgroups; the launch takes ceil(units / slots) rounds of
// one unit's time, the reduction reads splits * M * N * 4 bytes at about 4 TB/s.
static inline SplitKPlan splitk_plan(int64_t batch, int64_t m, int64_t n, int64_t k, double* model = nullptr) {
  SplitKPlan p{0, 0, 0.0};
  if (batch != 1 || k < 2048 || k % 32 != 0 || n <= 64 || m < 1) return p;
  const int64_t t128 = ((m + 127) / 128) * ((n + 127) / 128);
  if (t128 >= 256) return p;  // at least one tile per CU: no split
  const int64_t t256 = ((m + 255) / 256) * ((n + 255) / 256);
  double best = 0.0;
  for (int tile = 128; tile <= 256; tile += 128) {
    const int bk = tile == 128 ? 32 : 64;
    if (k % bk != 0) continue;
    if (tile == 256 && (m <= 128 || n <= 128)) continue;
    const int64_t tiles = tile == 128 ? t128 : t256;
    const int64_t slots = tile == 128 ? 512 : 256;
    const double unit_rate = tile == 128 ? 900e6 / 512 : 1240e6 / 256;  // FLOP per us per workgroup
    for (int64_t splits = 2; splits <= 16; ++splits) {
      if (k / bk / splits < 8) break;  // at least 8 stages per split
      const double chunk = static_cast<double>(k) / splits;
      // (a 128-tile workgroup that has its CU to itself runs about 1.7 times faster than one of
      // two: 768 x 768 x 16384 in 5 splits of 36 tiles takes 32 us)
      const double alone = (tile == 128 && tiles * splits <= 256) ? 1.7 : 1.0;
      const double unit = 2.0 * tile * tile * chunk / (unit_rate * alone);
      const double rounds = static_cast<double>((tiles * splits + slots - 1) / slots);
      const double reduce = 3.0 + static_cast<double>(splits) * m * n * 4.0 / 4e6;
      const double cost = rounds * unit + reduce;
      if (p.splits == 0 || cost < best) {
        best = cost;
        p.splits = static_cast<int>(splits);
        p.tile = tile;
      }
    }
  }
  if (model != nullptr) *model = best;
  return p;
}
// The same, or no split where one round of the tiles above is faster (the model's costs are 4.5 us under the measured ones).
// A row-major up to K = 4096, as far as their cost was fitted: 2100 x 768 x 3072 30.0 us split and 18.7, 4300 x 768 x 3072
// 45.2 and 33.7, 2000 x 768 x 3072 27.7 and 17.1, 3072 x 768 x 4096 42.4 and 32.3; 70 shapes of K 3072 .. 4096 take 0.79 of
// the time (geometric mean, worst 1.05). Beyond, the costs of both choose no better than the split (0.97 of the time, worst
// 1.16, over 350 shapes of K 4160 .. 8192). A stored [K, M] 3072 x 768 x 2048 27.5 and 19.3, x 4096 46 and 34, with half of
// the CUs idle level (2304 x 768 x 3072 24 both) or behind (224 x 7464 x 3008 29 and 35).
static inline SplitKPlan splitk_or_whole(int64_t batch, int64_t m, int64_t n, int64_t k, int trans_a) {
  double split_cost = 0.0;
  const SplitKPlan p = splitk_plan(batch, m, n, k, &split_cost);
  const int form = ring_one_round(batch, m, n, k, trans_a);
  if (p.splits == 0 || form == 0) return p;
  const int64_t t128 = ((m + 127) / 128) * ((n + 127) / 128);
  const bool whole = trans_a ? k < 2560 || (k <= 4096 && t128 > 128) : k <= 4096;
  return whole && one_round_cost(form, t128, k) < split_cost + 4.5 ? SplitKPlan{0, 0, 0.0} : p;
}

// fp32: microseconds of a launch on one of the kernels' tiles: a start and, per round of the 256 CUs, `per_k` for each k of
// a run and `per_tile` for the tile's way out, `edge` of which is stores that a tile past the matrix's edge leaves out;
// `whole` of a round's time is bound to whole rounds, and from eight rounds on time is linear in them. No less than all
// stores at 5.5 TB/s. Fitted to 165000 launches of 28800 shapes: 4 .. 16384 rows and columns, some 50257, K 4 .. 12000, 1 .. 64
// batches, all layouts. Off by 7 .. 17 % (rms) for each tile, most of which is the layout; what they choose is behind the
// best tile and split by 1.1 % on average.
struct F32Tile {
  int bm, bn, waves;
  double start, per_k, per_tile, power, whole, edge;
};
static inline double f32_tile_cost(const F32Tile& t, double copies, int64_t m, int64_t n, double run) {
  const double tiles = static_cast<double>(((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn)) * copies, r = tiles / 256.0;
  const double outputs = copies * static_cast<double>(m) * static_cast<double>(n);
  const double some = r < 8.0 ? r : 8.0;
  const double rounds = r <= 1.0 ? 1.0 : std::pow(some, t.power) * (r / some) * (1.0 - t.whole + t.whole * std::ceil(r) / r);
  const double per_tile = t.per_tile * (1.0 - t.edge + t.edge * outputs / (tiles * t.bm * t.bn));
  return std::fmax(t.start + rounds * (t.per_k * run + per_tile), 3.0 + outputs * 4.0 / 5.5e6);
}
// The second launch of a split product.
static inline double f32_reduction_cost(int64_t m, int64_t n, int splits) {
  return 3.6 + 0.8e-6 * splits * static_cast<double>(m) * static_cast<double>(n);
}
// Of the kernel whose waves share K. A 64 x 64 tile has eight waves where all tiles run at once (two a SIMD to hide each
// other's waits: 1332 x 768 x 3072 57 us, with four 70), four, two workgroups to a CU, beyond (1332 x 3072 x 768 58 us, with
// eight 66), and a 32 x 32 tile likewise (64 x 768 x 768 7.9 us, with four 9.2).
// (The two of eight waves are moved by 0.2 us of the fit, within its error: 128 x 768 x 3072 takes 17.2 us in two splits of
// 32 x 32 tiles and 17.4 in eight of 64 x 64, and keeps the latter.)
constexpr F32Tile kF32Tiles[] = {{32, 32, 4, 3.28, 0.00836, 0.837, 0.836, 0.49, 0.0},
                                 {32, 64, 4, 3.73, 0.0133, 2.08, 0.885, 0.48, 0.0},
                                 {64, 64, 4, 4.13, 0.0210, 3.34, 0.879, 0.49, 0.10},
                                 {64, 64, 8, 3.0, 0.0156, 4.2, 1.0, 0.0, 0.12}};
constexpr int kF32TileCount = sizeof(kF32Tiles) / sizeof(kF32Tiles[0]);
constexpr F32Tile kF32AllAtOnce = {32, 32, 8, 2.9, 0.0063, 1.2, 1.0, 0.0, 0.35};
// Short K runs with fp32 products, on 32 x 32 tiles only: 32 x 64 and 64 x 64 ones were faster by more than 3 % in 0.2 and 1 %
// of 10900 such launches.
constexpr F32Tile kF32Products = {32, 32, 4, 2.97, 0.00352, 0.746, 1.0, 0.68, 0.10};
struct F32Plan {
  int tile;    // index into kF32Tiles
  int splits;  // 0: not split
  double cost;
};
static inline double f32_cost(int tile, int64_t batch, int64_t m, int64_t n, int64_t k, int splits) {
  const double copies = static_cast<double>(splits > 0 ? splits : batch);
  const double run = static_cast<double>(k) / (splits > 0 ? splits : 1);
  const F32Tile& t = kF32Tiles[tile];
  const bool at_once = static_cast<double>(((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn)) * copies <= 256.0;
  if (k <= kF32SplitK) return tile == 0 ? f32_tile_cost(kF32Products, copies, m, n, run) : HUGE_VAL;
  if (t.bm == 64 && at_once != (t.waves == 8)) return HUGE_VAL;
  return f32_tile_cost(t.bn == 32 && at_once ? kF32AllAtOnce : t, copies, m, n, run);
}
static inline F32Plan f32_plan(int64_t batch, int64_t m, int64_t n, int64_t k, int most_splits) {
  F32Plan p{0, 0, HUGE_VAL};
  for (int i = 0; i < kF32TileCount; ++i) {
    const double c = f32_cost(i, batch, m, n, k, 0);
    if (c < p.cost) p = F32Plan{i, 0, c};
  }
  if (batch != 1 || m * n >= (int64_t{1} << 31)) return p;
  double best = p.cost * 0.95;  // a second launch and a workspace have to pay for themselves
  for (const int s : {2, 3, 4, 6, 8, 12, 16}) {
    if (k < 96 * s || s > most_splits) break;
    for (int i = 0; i < kF32TileCount; ++i) {
      const double c = f32_cost(i, 1, m, n, k, s) + f32_reduction_cost(m, n, s);
      if (c < best) {
        best = c;
        p = F32Plan{i, s, c};
      }
    }
  }
  return p;
}
// The kernel of 128 x 128 tiles, and the one with fp32 products that takes its place at short K.
constexpr F32Tile kF32WideTile = {128, 128, 8, 2.32, 0.0450, 6.57, 1.07, 1.0, 0.48};
constexpr F32Tile kF32WideProducts = {128, 128, 4, 1.89, 0.0775, 4.46, 0.869, 0.74, 0.59};
static inline double f32_wide_cost(int64_t batch, int64_t m, int64_t n, int64_t k, int splits) {
  const double copies = static_cast<double>(splits > 0 ? splits : batch);
  return f32_tile_cost(k <= kF32SplitK ? kF32WideProducts : kF32WideTile, copies, m, n,
                       static_cast<double>(k) / (splits > 0 ? splits : 1));
}
// Operands off 16-byte boundaries are as fast there (its loads want none), and run there from this K on; shorter products
// of such operands are the padded copies', the vector kernel's and the waves-share-K kernel's.
constexpr int64_t kF32WideUnalignedK = 512;
struct F32WidePlan {
  bool taken;  // before the kernel whose waves share K
  int splits;
  double cost;
};
// Where a product whose operands both take runs on it (`other`: what it runs as otherwise), and with how many splits. Up to
// 40 tiles only: callers rely on products that fill most CUs with 64 x 64 tiles to ask for no scratch (1024 x 768 x 3072, 48
// tiles). Splitting on would pay: 1024 x 768 x 3072 58 us unsplit, 47 in five runs, 2048 x 768 x 3072 99 and 83.
constexpr int64_t kF32WideSplitTiles = 40;
static inline F32WidePlan f32_wide_plan(int64_t batch, int64_t m, int64_t n, int64_t k, const F32Plan& other) {
  F32WidePlan p{false, 0, f32_wide_cost(batch, m, n, k, 0)};
  p.taken = p.cost < other.cost;
  if (batch != 1 || m * n >= (int64_t{1} << 31) || ((m + 127) / 128) * ((n + 127) / 128) > kF32WideSplitTiles) return p;
  double best = (p.taken ? p.cost : other.cost) * 0.95;  // (as above)
  for (int s = 2; s <= 16 && k >= 96 * s; ++s) {
    const double c = f32_wide_cost(1, m, n, k, s) + f32_reduction_cost(m, n, s);
    if (c < best) {
      best = c;
      p = F32WidePlan{true, s, c};
    }
  }
  return p;
}
// Unaligned operands: the other way is to copy what the 128 x 128 kernel cannot read into padded buffers (6 us a copy
// with what the host does for it, and the bytes at 5.3 TB/s, 1.3 where it transposes) and to multiply there, a K that is no
// whole number of 16-byte vectors as the next multiple of 64; infinite where the copies would not run on that kernel.
// 3072 x 4096 x 97 48 us, 58 where it lies; 3072 x 2048 x 97 35 and 29.
// 7710 x 8280 x 8 60 against 317 us where it lies, 48 x 816 x 3664 x 16 175 against 721, 8051 x 6756 x 172 with a
// residual 350 against 630.
static inline double f32_padded_cost(int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, bool a_ok,
                                     bool b_ok, int trans_a, int trans_b) {
  double cost = 0.0;
  auto copy = [&](int64_t elements, bool transposing) {
    cost += 6.0 + static_cast<double>(elements) * batch * 8.0 / (transposing ? 1.3e6 : 5.3e6);
  };
  int64_t depth = k;
  const bool b_fits = b_ok && ldb % 4 == 0;
  if (trans_a && batch == 1 && b_fits && (trans_b ? k : n) % 4 == 0) {
    copy(m * k, false);  // (zero columns; it stays transposed)
  } else {
    depth = k % 4 == 0 ? k : (k + 63) / 64 * 64;
    if (trans_a) copy(m * k, true);
    if (depth != k || (!trans_a && (lda % 4 != 0 || !a_ok))) copy(m * k, false);
    if (!trans_b && b_fits && n % 4 == 0) {
      if (depth != k) copy(n * k, false);
    } else if (!(trans_b && b_fits && depth == k)) {
      copy(n * k, !trans_b);
    }
  }
  const F32WidePlan wide = f32_wide_plan(batch, m, n, depth, f32_plan(batch, m, n, depth, 16));
  return wide.taken && wide.splits == 0 ? cost + wide.cost : HUGE_VAL;
}
// What the kernel whose waves share K asks of its operands: at least four elements along each contiguous direction, and
// lane offsets that fit 32 bits in its largest tile (64 x 64, of which B is held to twice the rows; 32 rows of k for an
// operand stored K-outer).
static inline bool f32_shared_eligible(const GemmArgs& g, int trans_a, int trans_b) {
  if (g.m < 1 || g.n < 1 || g.k < 1) return false;
  if ((trans_a ? g.m : g.k) < 4 || (trans_b ? g.k : g.n) < 4) return false;
  auto reached = [](int64_t lines, int64_t ld) { return ld < ((int64_t{1} << 30) - 256) / (lines > 1 ? lines - 1 : 1); };
  return reached(trans_a ? kF32KS : (g.m < 64 ? g.m : 64), g.lda) &&
         reached(trans_b ? (g.n < 128 ? g.n : 128) : kF32KS, g.ldb);
}

// Which kernel takes a product, with its tile (an index into the kernel's own list) and
// its number of splits (0: not split). The launch follows it (gemm_typed.h), and tmb_gemm_route answers it.
struct GemmRoute {
  int kernel;  // TMB_GEMM_*, or TMB_ERR_UNSUPPORTED
  int tile;
  int splits;
};

static inline GemmRoute route_16bit(const GemmArgs& g, int64_t batch, int trans_a, int trans_b, int epilogue,
                                    size_t workspace_bytes) {
  if (g.residual != nullptr && g.round_like_unfused) {
    // the bits of the product alone, rounded, and an add: the kernel, tile and splits that it runs on by itself, or none
    GemmArgs alone = g;
    alone.residual = nullptr;
    GemmRoute r = route_16bit(alone, batch, trans_a, trans_b, epilogue, workspace_bytes);
    if (r.kernel == TMB_GEMM_STREAM64 && mfma_eligible(g, batch, trans_a, trans_b))
      r.kernel = TMB_GEMM_RING;  // (adds its four steps of K in the same order)
    // (a transposed A that one round of the rings takes in place of a split launch: added where that launch's reduction did,
    // by the tiles' way out)
    if (r.kernel == TMB_GEMM_TRANSPOSED_A) {
      const int splits = splitk_plan(batch, g.m, g.n, g.k).splits;
      if (splits > 0 && workspace_bytes >= static_cast<size_t>(splits) * g.m * g.n * 4) return r;
    }
    if (r.kernel == TMB_GEMM_TRANSPOSED_A || r.kernel == TMB_GEMM_STREAM64 || r.kernel == TMB_GEMM_SIMT)
      return {TMB_ERR_UNSUPPORTED, 0, 0};
    return r;
  }
  const bool aligned = mfma_eligible(g, batch, trans_a, trans_b);
  const bool whole_columns = trans_b || g.n % 8 == 0;
  if (aligned && whole_columns && small_applies(batch, g.m, g.n, g.k))
    return {TMB_GEMM_SMALL, small_tile(batch, g.m, g.n, g.k), 0};
  if (workspace_bytes > 0) {
    // (a transposed A with a residual or a GELU: the reduction takes them along, the rings do not, but for a GELU that is to
    // have the bits of two operations, on the tiles that the product alone runs on)
    const bool gelu_after = trans_a && epilogue != TMB_EPI_NONE;
    const bool split_only = trans_a && (g.residual != nullptr || (gelu_after && !g.round_like_unfused));
    const SplitKPlan split = splitk_plan(batch, g.m, g.n, g.k);
    const SplitKPlan plan = split_only ? split : splitk_or_whole(batch, g.m, g.n, g.k, trans_a);
    const bool operands_ok = trans_a ? mfma_transposed_a_eligible(g, batch, trans_a, trans_b, TMB_EPI_NONE)
                                     : aligned && whole_columns;
    if (split.splits > 0 && operands_ok && g.m * g.n < (int64_t{1} << 31) &&
        workspace_bytes >= static_cast<size_t>(split.splits) * g.m * g.n * 4) {
      if (plan.splits > 0) return {TMB_GEMM_SPLITK, plan.tile == 256 ? 1 : 0, plan.splits};
      if (gelu_after) return {TMB_GEMM_TRANSPOSED_A, 0, 0};
    }
  }
  if (g.residual == nullptr && mfma_transposed_a_eligible(g, batch, trans_a, trans_b, epilogue))
    return {TMB_GEMM_TRANSPOSED_A, 0, 0};
  // (in front of the any-layout kernel: it takes operands beyond the rings' 4 GiB)
  if (!trans_a && stream64_eligible(g, batch, trans_b, epilogue)) return {TMB_GEMM_STREAM64, 0, 0};
  if (!aligned && any_eligible(g.m, g.n, g.k, g.lda, g.ldb, trans_a, trans_b)) {
    AnyPlan plan = any_plan(batch, g.m, g.n, g.k, true);
    if (plan.splits > 0 && workspace_bytes < static_cast<size_t>(plan.splits) * g.m * g.n * 4)
      plan = any_plan(batch, g.m, g.n, g.k, false);
    if (g.residual != nullptr && mfma_transposed_a_eligible(g, batch, trans_a, trans_b, epilogue) &&
        !any_with_residual_pays(g, batch, plan.cost))
      return {TMB_ERR_UNSUPPORTED, 0, 0};
    if (simt_instead_of_any(g, batch, plan)) return {TMB_GEMM_SIMT, 0, 0};
    return {TMB_GEMM_ANY, plan.tile, plan.splits};
  }
  if (aligned) return {TMB_GEMM_RING, 0, 0};
  if (g.residual != nullptr) return {TMB_ERR_UNSUPPORTED, 0, 0};
  return {TMB_GEMM_SIMT, 0, 0};
}

// A residual is carried where the product alone runs on the kernel whose waves share K or on a split launch, whose
// reduction adds it, and added by the caller where it does not: the sum has the bits of the two operations, and carrying it
// saves next to nothing on the others (2 us a million elements there, as much as the add).
static inline GemmRoute route_f32(const GemmArgs& g, int64_t batch, int trans_a, int trans_b,
                                  size_t workspace_bytes) {
  if (g.residual != nullptr) {
    GemmArgs alone = g;
    alone.residual = nullptr;
    const GemmRoute r = route_f32(alone, batch, trans_a, trans_b, workspace_bytes);
    const bool carried = r.kernel == TMB_GEMM_F32 ||
                         (r.kernel == TMB_GEMM_F32_WIDE && r.splits > 0 && f32_shared_eligible(g, trans_a, trans_b));
    return carried ? r : GemmRoute{TMB_ERR_UNSUPPORTED, 0, 0};
  }
  const bool shared = f32_shared_eligible(g, trans_a, trans_b);
  const bool aligned = f32_mfma_eligible(g, batch, trans_a, trans_b);
  if (!shared && !aligned) return {TMB_GEMM_SIMT, 0, 0};
  auto fits = [&](int splits) {
    return splits == 0 || workspace_bytes >= static_cast<size_t>(splits) * g.m * g.n * 4;
  };
  if (shared) {
    F32Plan plan = f32_plan(batch, g.m, g.n, g.k, 16);
    const F32WidePlan wide = f32_wide_plan(batch, g.m, g.n, g.k, plan);
    const bool takes = aligned || g.k >= kF32WideUnalignedK;
    if (takes && wide.taken && fits(wide.splits)) return {TMB_GEMM_F32_WIDE, 0, wide.splits};
    // (no more splits than there: the scratch that a caller of known layout is told of does not depend on alignment)
    if (wide.splits > 0 && plan.splits > wide.splits) plan = f32_plan(batch, g.m, g.n, g.k, wide.splits);
    if (!fits(plan.splits)) plan = f32_plan(batch, g.m, g.n, g.k, 0);
    if (takes && plan.splits == 0 && f32_wide_cost(batch, g.m, g.n, g.k, 0) < plan.cost)
      return {TMB_GEMM_F32_WIDE, 0, 0};
    if (g.k <= 48 && plan.splits == 0 && simt_cost(true, batch, g.m, g.n, g.k) < plan.cost) return {TMB_GEMM_SIMT, 0, 0};
    return {TMB_GEMM_F32, plan.tile, plan.splits};
  }
  // rows too long for 32-bit offsets: the wide kernel, which addresses in 64 bits, split as far as the other one would be
  const int splits = f32_plan(batch, g.m, g.n, g.k, 16).splits;
  return {TMB_GEMM_F32_WIDE, 0, fits(splits) ? splits : 0};
}

// The most splits that a product of dense operands in this layout runs with, at any alignment.
static inline int f32_most_splits(int64_t batch, int64_t m, int64_t n, int64_t k, int trans_a, int trans_b) {
  int most = 0;
  for (const uintptr_t address : {16, 20}) {  // (never read: only their alignment is looked at)
    GemmArgs g{};
    g.a = g.b = reinterpret_cast<const void*>(address);
    g.m = m, g.n = n, g.k = k;
    g.lda = trans_a ? m : k, g.ldb = trans_b ? k : n;
    g.stride_a = m * k, g.stride_b = k * n;
    const int splits = route_f32(g, batch, trans_a, trans_b, ~size_t{0}).splits;
    most = splits > most ? splits : most;
  }
  return most;
}

// The typed half of the entry point (gemm_typed.h), one translation unit per storage type.
template <typename T>
int gemm_epi(const GemmArgs& g, int64_t batch, int ta, int tb, int epilogue, hipStream_t stream, void* ws,
             size_t ws_bytes);

}  // namespace tmb
