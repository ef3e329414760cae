// Which tile a W4A16 or scaled fp8 product runs on: host-only C++ (no HIP),
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

// The tile of a dense product of more than 16 rows, by the same estimate (us per
// K step, measured at K = 4096 and 11008 on 43 - 1376 tiles).  Up to 64 rows
// 64-column tiles of four K groups put a product on every CU that has columns
// for it: 48 rows x 11008 columns 15 us against 25 (64 x 128), 30 (64 x 256)
// and 62 (256 x 256).  128 x 11008 (K = 4096): 64 x 128 25 us, 64 x 256 31, 128
// x 256 42, 256 x 256 63; 512 x 11008: 61 / 59 / 52 / 71; 1024 x 11008: 116 /
// 101 / 106 / 95; 500 x 4096 (K = 11008): 65 / 78 / 106 / 160.
inline DenseTile pick_dense_tile(int64_t M, int64_t N) {
  auto tiles = [&](int64_t tm, int64_t tn) { return (double)((M + tm - 1) / tm * ((N + tn - 1) / tn)) / 256.0; };
  // x: tiles per CU
  auto c64 = [](double x) { return 0.18 * std::max(1.0, x); };
  auto c128 = [](double x) { return x <= 1 ? 0.30 + 0.05 * x : std::max(0.5, 0.32 * x); };
  auto c256 = [](double x) { return x <= 1 ? 0.40 + 0.10 * x : std::max(0.83, 0.55 * x); };
  auto c128x256 = [](double x) { return x <= 1 ? 0.56 + 0.25 * x : std::max(1.56, x); };  // one tile per CU
  auto cbig = [](double x) { return x <= 1 ? 0.80 + 0.85 * x : std::max(2.66, 1.74 * x); };
  DenseTile best = DENSE_256;
  double c = cbig(tiles(256, 256));
  auto take = [&](DenseTile t, double cost) {
    if (cost < c) best = t, c = cost;
  };
  take(DENSE_128x256, c128x256(tiles(128, 256)));
  take(DENSE_64x256, c256(tiles(64, 256)));
  take(DENSE_64x128, c128(tiles(64, 128)));
  if (M <= 64) take(DENSE_64x64_K4, c64(tiles(64, 64)));
  return best;
}

// Rows per block of the few-row scaled fp8 GEMM (32, 64 or 128; 32 columns per
// block), or 0 for the 256 x 256 tiles.  A few-row block is bound by its CU's
// loads: measured about 1.5 us + (its rows of A and W) x K / 33 KB per us, blocks
// that share a CU in turn (8192 x 8192 weights: 1 row 12.4 us, 32 rows 17.4, 64
// rows 24.6 in 64-row blocks and 31.6 in 32-row ones; 128 x 4096 x 4096: 17.8 /
// 14.1 / 21.9 us in 32- / 64- / 128-row blocks).  A round of 256 x 256 tiles takes
// 5 us + 0.9 us per 128 bytes of K on a few CUs, 1.55 us on all (block scales:
// 1.45 and 1.9): 32 rows 65 us, 256 x 4096 x 4096 38 us (few-row 22.5), 512 x 4096
// x 4096 39 us (few-row 40).
inline int pick_fp8_rows(int64_t M, int64_t N, int64_t K, bool block_scaled) {
  const double steps = (double)K / 128;
  const double x = (double)((M + 255) / 256 * ((N + 255) / 256)) / 256;
  const double few = block_scaled ? 1.45 : 0.9, all = block_scaled ? 1.9 : 1.55;
  double c = x <= 1 ? 5 + steps * (few + (all - few) * x) : (5 + steps * all) * x;
  int best = 0;
  for (int rows : {32, 64, 128}) {
    const double blocks = (double)((M + rows - 1) / rows * ((N + 31) / 32));
    const double rounds = (double)(int64_t)((blocks + 255) / 256);
    const double t = rounds * (1.5 + (double)(std::min<int64_t>(rows, M) + 32) * (double)K / 33e3);
    if (t < c) best = rows, c = t;
  }
  return best;
}

}  // namespace plan
}  // namespace tb
