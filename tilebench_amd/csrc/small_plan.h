// Which tile a W4A16, scaled fp8 or plain product runs on: host-only C++ (no HIP),
// shared with a CPU check.
//
// A W4A16 product's time is about its K steps times the time of one step of all its
// tiles on 256 CUs.  Measured on MI355X (graph replays, K = 4096, us per K step
// of 64): a 32 x 128 tile takes 0.25, 32 x 256 0.37, 64 x 256 0.42 - 0.56 (one
// tile per CU - many), 256 x 256 0.9 - 1.9 (its MFMAs at the power cap).  Tiles
// that share a CU share its VALU (the dequantisation bounds the small ones), so
// their steps add up; a 256 x 256 tile fills a CU.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace tb {
namespace plan {

enum ExpertTile { TILE_256 = 0, TILE_32x128, TILE_32x256, TILE_64x256 };

// Tiles of `tm` rows for `rows` rows over `active` experts: half a tile of
// padding per expert, at least one tile each.
inline double expert_tile_rows(double rows, double active, double tm) {
  return std::max(active, rows / tm + active / 2);
}

// The tile of a grouped, gate/up (N = 2 I columns of W13) or down product.  The
// host knows the row count only, so at most `rows` experts have a tile and the
// rows are taken as spread over them.  Measured (64 experts, top 8, H = 4096, I =
// 704; gate/up + down us, this tile against 256 x 256): 1 token 23 + 8 (32 x
// 128) against 84 + 18; 24 tokens 48 + 20 (32 x 256) against 164 + 56; 256
// tokens 68 + 33 (64 x 256, 32 x 256) against 166 + 69; 1024 tokens 137 + 74
// (64 x 256) against 191 + 104; 4096 tokens 445 + 265 (64 x 256) against 414 +
// 251: the 256-row tiles stay there.
inline ExpertTile pick_expert_tile(int64_t rows, int64_t experts, int64_t N) {
  const double r = (double)rows, active = (double)std::min(rows, experts);
  const double n128 = (double)((N + 127) / 128), n256 = (double)((N + 255) / 256);
  const double big_n = (double)((N + 127) / 128) / 2;  // a last column tile of <= 128 columns is half a tile
  auto load = [](double tiles) { return std::max(1.0, tiles / 256.0); };
  const double c128 = 0.25 * load(expert_tile_rows(r, active, 32) * n128);
  const double c256 = 0.37 * load(expert_tile_rows(r, active, 32) * n256);
  const double tiles64 = expert_tile_rows(r, active, 64) * n256;
  const double c64 = tiles64 <= 256 ? 0.42 + 0.14 * tiles64 / 256 : 0.56 * tiles64 / 256;
  const double tiles_big = expert_tile_rows(r, active, 256) * big_n;
  const double cbig = tiles_big <= 256 ? 0.9 : std::max(1.8, 1.88 * tiles_big / 256);
  ExpertTile best = TILE_256;
  double c = cbig;
  if (c64 < c) best = TILE_64x256, c = c64;
  if (c256 < c) best = TILE_32x256, c = c256;
  if (c128 < c) best = TILE_32x128, c = c128;
  return best;
}

enum DenseTile { DENSE_256 = 0, DENSE_64x64_K4, DENSE_64x128, DENSE_64x256, DENSE_128x256 };

// us of a K step of `x` tiles per CU, as it was measured: a line over the first
// round of tiles, then a stair per round (a round that is nearly empty costs nearly
// as much as a full one) with a slope for how full the last one is.  `power` is for
// the 256 x 256 tiles, whose clock falls with the share of the chip that multiplies
// (`work`: tiles per CU without their padding).
struct Stairs {
  double first, slope, second, round, fill, power = 0;
  double operator()(double x, double work = 0) const {
    if (x <= 1) return first + slope * x + power * std::max(0.0, work - 0.3);
    const double rounds = std::ceil(x);
    return second + round * (rounds - 2) + fill * (x - (rounds - 1));
  }
};

// The tile of a dense product of more than 16 rows, by the same estimate.  The
// constants are least-squares fits over sizes of 17 - 8192 rows, K and N 64 - 32768 (cold
// weights, each tile forced in turn): within 7 % of nine in ten.  The 256 x 256
// tiles are priced 2 % below their fit, so that a tie goes to them.  Over 5177 sizes the
// picks then took 0.2 % more than the best tile, and two over 3 % more than 256 x 256
// (636 x 28552, K 2368: 102 us against 97).
// Up to 64 rows 64-column tiles of four K groups put a product on every CU that has
// columns for it: 48 rows x 11008 columns 15 us against 25 (64 x 128), 30 (64 x 256)
// and 62 (256 x 256); up to 32 rows the launch halves its rows (12.5 at 32 rows,
// 13.9 on 64).  500 x 4096 (K = 11008): 64 x 128 65 us, 64 x 256 78, 128 x 256 106,
// 256 x 256 160.  Half a round of 256 x 256 tiles beats two rounds and a bit of any
// smaller one: 729 x 12288 (K = 4096) 72 us against 91 (64 x 256), 2391 x 3608 (K =
// 10560) 193 against 247 (128 x 256).
inline DenseTile pick_dense_tile(int64_t M, int64_t N) {
  auto tiles = [&](int64_t tm, int64_t tn) { return (double)((M + tm - 1) / tm * ((N + tn - 1) / tn)) / 256.0; };
  constexpr double steps = 64;  // K = 4096: the start and end of a tile weigh little beside its steps
  constexpr Stairs s64{0.11, 0.20, 0.62, 0.25, 0}, s128{0.30, 0.07, 0.48, 0.33, 0.18},
      s256{0.41, 0.15, 0.82, 0.56, 0.26}, s128x256{0.56, 0.30, 1.49, 1.02, 0.38},
      sbig{0.86, 0.26, 2.40, 1.77, 0.83, 0.72};
  DenseTile best = DENSE_256;
  double c = 0.98 * (6 + steps * sbig(tiles(256, 256), (double)M * (double)N / 65536.0 / 256.0));
  auto take = [&](DenseTile t, double cost) {
    if (cost < c) best = t, c = cost;
  };
  take(DENSE_128x256, 5 + steps * s128x256(tiles(128, 256)));
  take(DENSE_64x256, 4 + steps * s256(tiles(64, 256)));
  take(DENSE_64x128, 4 + steps * s128(tiles(64, 128)));
  if (M <= 64) take(DENSE_64x64_K4, 4 + steps * s64(tiles(64, 64)));
  return best;
}

enum Fp8Tile { FP8_256 = 0, FP8_32x32, FP8_64x64, FP8_64x128, FP8_128x128 };

// The tile of a scaled fp8 product, by estimated time in us (s: steps of 128
// bytes of K, x: tiles per CU; measured with s = 8 - 64).  32 x 32 blocks are
// bound by their CU's loads, 1.5 us + (rows of A and W) x K / 33 KB per us, and
// run in rounds of 256; a step of the LDS tiles takes 0.2 us at 64 x 64, 0.31
// at 64 x 128 (block scales 0.34), 0.36 - 0.5 at 128 x 128 (0.42 - 0.57), and tiles
// that share a CU share its LDS.  A step of 256 x 256 tiles takes 0.9 us on a few
// CUs and 1.55 us on all (1.45 and 1.9).
// Measured, these tiles against 256 x 256 (us): 1 x 8192 x 8192 12 / 65 (32 x 32),
// 64 x 8192 x 8192 15 / 66, 200 x 2112 x 7168 13 / 60 and 14 / 88 (64 x 64), 256 x
// 8192 x 8192 25 / 69 (64 x 128), 512 x 8192 x 8192 35 / 69, 1024 x 4096 x 4096 23 /
// 40, 1024 x 8192 x 8192 60 / 76 (128 x 128); 1348 x 7168 x 4224 56 / 46,
// block scales 4096 x 2112 x 7168 98 (64 x 128) / 92: the 256 x 256 tiles stay.
inline Fp8Tile pick_fp8_tile(int64_t M, int64_t N, int64_t K, bool block_scaled) {
  const double s = (double)K / 128;
  auto tiles = [&](int64_t tm, int64_t tn) { return (double)((M + tm - 1) / tm * ((N + tn - 1) / tn)) / 256.0; };
  auto up = [](double v) { return (double)(int64_t)(v + 0.999999); };
  const double few = block_scaled ? 1.45 : 0.9, all = block_scaled ? 1.9 : 1.55;
  const double big = tiles(256, 256);
  double c = big <= 1 ? 5 + s * (few + (all - few) * big) : (5 + s * all) * big;
  Fp8Tile best = FP8_256;
  auto take = [&](Fp8Tile t, double cost) {
    if (cost < c) best = t, c = cost;
  };
  const double t128 = tiles(128, 128);
  if (t128 <= 1)
    take(FP8_128x128, 3 + s * (block_scaled ? 0.42 + 0.15 * t128 : 0.36 + 0.14 * t128));
  else
    take(FP8_128x128, up(t128 / 2) * (3 + s * (block_scaled ? 1.04 : 0.95)));
  const double t64x128 = up(tiles(64, 128)), t64 = up(tiles(64, 64));
  take(FP8_64x128, 3 * std::max(1.0, t64x128 / 2) + s * (block_scaled ? 0.34 * t64x128 : 0.30 * t64x128 + 0.03));
  take(FP8_64x64, 3 * std::max(1.0, t64 / 2) + s * std::max(0.20, 0.19 * t64));
  take(FP8_32x32, up(tiles(32, 32)) * (1.5 + (double)(std::min<int64_t>(32, M) + 32) * (double)K / 33e3));
  return best;
}

enum NtTile { NT_256 = 0, NT_64x64, NT_64x128, NT_128x128 };

// The tile of a plain product (Kb: bytes of K per operand row), by the same
// estimate: a step of 128 bytes takes 0.2 us at 64 x 64, 0.31 at 64 x 128, 0.36 -
// 0.54 at 128 x 128 (two of them share a CU and step in 0.75 - 1.1, not in twice that)
// and 1.35 - 1.95 at 256 x 256, whose start and end take 4 us more than a small tile's
// (fp16 and fp32; the others within a fifth).  Over 3018 sizes of the four types the picks
// take 0.3 % more than the best tile; without those two terms fp32 3380 x 1192 x 3968 ran
// on 64 x 64 tiles (177 us, 128 x 128 156) and int8 2779 x 3616 x 256 on 256 x 256
// (22.7, 128 x 128 19.6).  Measured fp16 products alone, us: 16 x 4096 x 4096 14.7 (64 x 64;
// 256 x 256 86), 512 x 4096 x 4096 23.4 (64 x 128; 93), 2048 x 2048 x 4096 39 (128 x
// 128; 95), 2601 x 1648 x 2432 30 (128 x 128; 58), 2872 x 3104 x 5504 with its
// transpose 155 (128 x 128; 256 x 256 158), 4096 x 4096 x 4096 129 (256 x 256; 128 x 128 135).
inline NtTile pick_nt_tile(int64_t M, int64_t N, int64_t Kb) {
  const double s = (double)Kb / 128;
  auto tiles = [&](int64_t tm, int64_t tn) { return (double)((M + tm - 1) / tm * ((N + tn - 1) / tn)) / 256.0; };
  auto up = [](double v) { return (double)(int64_t)(v + 0.999999); };
  const double big = tiles(256, 256), t128 = tiles(128, 128), t64x128 = up(tiles(64, 128)), t64 = up(tiles(64, 64));
  double c = 4 + 3 * std::max(1.0, big) + s * (big <= 1 ? 1.35 + 0.2 * big + std::max(0.0, big - 0.6) : 1.95 * big);
  NtTile best = NT_256;
  auto take = [&](NtTile t, double cost) {
    if (cost < c) best = t, c = cost;
  };
  constexpr Stairs s128{0.36, 0.18, 0.75, 0.65, 0.35};
  take(NT_128x128, 3 * std::max(1.0, up(t128) / 2) + s * s128(t128));
  take(NT_64x128, 3 * std::max(1.0, t64x128 / 2) + s * (0.30 * t64x128 + 0.03));
  take(NT_64x64, 3 * std::max(1.0, t64 / 2) + s * std::max(0.2, 0.19 * t64));
  return best;
}

constexpr int DEC_WAVES = 8, DEC_UNIT = 32, DEC_MAX_SPLITS = 16;
struct DecodePlan {
  int cols;       // columns of a slab, 128 or 256
  int64_t slabs;
  int splits;     // blocks that share a slab's K
};

// Slab width and K splits of the W4A16 decode kernel by an estimate of its time
// (us at M = 16): a wavefront takes its 32-row units one after the other, 0.75
// each at 128 columns and 1.45 at 256 (there a CU's stream binds: the mean share
// counts, not the longest; K 4096, N 12288 from cold 14.1 on 192 CUs, 13.4 on 240); a
// split costs an exchange of partials (1.5 or 3.6) that grows with the blocks taking
// part (0.55 or 0.6 each); and 128-column slabs, which read half lines, lose 0.09 per
// MB of weights and 0.2 more per MB above 23.  Fitted to 420 sizes, each with weights
// that stay in the last-level cache, that rotate through HBM, and that follow a fill of
// the cache with written lines: the picks take 0.2 - 0.3 % more than the better width, and 8
// of 2520 take over 3 % more than the 256-column kernel that was here before (worst 1 x
// 7184, K 6656, after a fill: 16.8 us against 15.3).  Measured, 128 / 256 columns at
// their best splits: K 4096, N 4096
// 7.8 / 11.4; K 4096, N 11008 11.9 / 12.5; K 4096, N 12288 14.4 / 12.9; K 8192, N
// 28672 43.1 / 32.6.  Splits at 128
// columns, K 4096, N 4096: 1 13.1, 2 9.7, 4 7.8, 8 8.5; K 1024, N 12288: 1 6.0, 2 6.7.
// A split grid never has more blocks than CUs, counted as they are launched: pairs of
// 128-column slabs go to the 8 XCDs in turn, and a block fills a CU, so a pair too many on
// one XCD would start its blocks a whole block's time later (9 x 6528, K 9920, five splits
// of 51 slabs, 34 blocks on an XCD of 32 CUs: 19.6 us; 256-column slabs 16.1, bounded 14.2).
inline int64_t decode_grid(int cols, int64_t slabs, int splits) {
  return cols == 128 ? ((slabs + 1) / 2 * splits + 7) / 8 * 16 : slabs * splits;
}

inline DecodePlan pick_decode(int64_t N, int64_t K, int cus) {
  const int64_t units = K / DEC_UNIT;
  const double mb = 0.5e-6 * (double)N * (double)K;  // of weights
  DecodePlan best{128, (N + 127) / 128, 1};
  double c = -1;
  for (int cols = 128; cols <= (N <= 128 ? 128 : 256); cols += 128) {  // the wide slab needs 16 columns
    const bool wide = cols == 256;
    const int64_t slabs = (N + cols - 1) / cols;
    for (int s = 1; s <= DEC_MAX_SPLITS && (s == 1 || (decode_grid(cols, slabs, s) <= cus && (int64_t)s * DEC_WAVES <= units)); ++s) {
      const double rounds = (double)((slabs * s + cus - 1) / cus), share = (double)units / (s * DEC_WAVES);
      double cost = wide ? rounds * std::max(1.0, share) * 1.45
                         : rounds * (double)(int64_t)(share + 0.999999) * 0.75 + 0.09 * mb + 0.2 * std::max(0.0, mb - 23);
      if (s > 1) cost += wide ? 3.6 + 0.6 * s : 2.1 + 0.55 * s;
      if (c < 0 || cost < c) best = DecodePlan{cols, slabs, s}, c = cost;
    }
  }
  return best;
}

}  // namespace plan
}  // namespace tb
