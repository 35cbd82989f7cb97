// q8_tiles.hpp -- which kernel and tile a Q8_0 linear takes: the measured costs
// and the choice among them, host code without HIP.
#pragma once
#include <cmath>
#include <cstdint>

namespace lux3d {

// Few: q8_0_few_rows_kernel, rows x 16 (rows 16: one row tile, 64: four);
// else a GEMM tile of rows x cols whose k is shared by `groups` groups of
// wavefronts.
struct Q8Tile {
  int rows, cols, groups;
  bool few() const { return cols == 16; }
};

inline double q8_tiles(int64_t m, int64_t n, int64_t bm, int64_t bn) {
  return (double)((m + bm - 1) / bm) * (double)((n + bn - 1) / bn);
}
inline double q8_rounds(double tiles) { return std::ceil(tiles / 256); }

// The few-rows kernel's grid: its row tiles are the launch's y, at most 65535.
constexpr int64_t kFewRowsMaxM = 65535 * 64;

// f32 activations: the kernel and tile that take the shortest time by these
// measured costs, linear in the 32-deep steps of k (ns; one round = every CU
// busy once, alone or, for the 64 x 128 tiles, with two workgroups):
//   few rows      64 x 16     262 steps + 2000 a round
//   1 x 4, KG 3   32 x 128    345 steps + 3500 a round
//   2 x 2, KG 2   64 x 128    570 steps + 4500 a round
//   2 x 2         64 x 128   1050 steps + 4000 for two a CU, 760 steps + 4000 for one
//   2 x 4        128 x 256   1500 steps + 5000 a round
// With 128 x 256 tiles alone a product of 1029 rows left most CUs idle or took
// a second round for a few tiles: 1029 x 4096 -> 1024 154 -> 76 us, 1029 x 1536
// -> 1536 76 -> 34, 512 x 8192 -> 2048 268 -> 91, 2049 x 1024 -> 4096 109 -> 91,
// 256 x 1024 -> 4096 36.7 -> 16.1. The share of `one` that the 64 x 128 tiles
// past a full round of 512 cost is fitted where it matters first, just past the
// round (model against measured: 516 tiles 85 / 87 us, 552 62 / 62, 1032 90 /
// 93, 1104 180 / 179); towards the next round it is up to a quarter too long
// (752 tiles 144 / 116), so that some sizes keep the 128 x 256 tile where this
// one is shorter (2500 x 1024 -> 4096: 111 us against 96), and none takes a
// longer one than before.
//
// Up to 16 rows one row tile of the few-rows kernel, whose time grows with the
// weights and, as every workgroup reads all of x, with m; a GEMM tile reads x
// once for 128 weight rows (us, few rows / 32 x 128 with three groups: 16 x
// 4096 -> 32000 100 / 50, 1 x 4096 -> 32000 61 / 47, 16 x 1024 -> 16384 15.0 /
// 14.8, 1 x 1024 -> 24576 13.4 / 14.9, 16 x 1024 -> 8192 8.8 / 14.7).
inline Q8Tile q8_tile_f32(int64_t m, int64_t n, int64_t k) {
  const double steps = (double)(k / 32), mid = q8_tiles(m, n, 64, 128);
  if (m <= 16) {
    const double one_tile = q8_tiles(m, n, 16, 16) / 256 * steps * (55 + 2.6 * (double)m) + 2000;
    if (0.96 * one_tile <= q8_rounds(q8_tiles(m, n, 32, 128)) * (300 * steps + 5300)) return {16, 16, 1};
    return {32, 128, 3};
  }
  const double few = m > kFewRowsMaxM ? INFINITY : q8_rounds(q8_tiles(m, n, 64, 16)) * (262 * steps + 2000);
  const double k3 = q8_rounds(q8_tiles(m, n, 32, 128)) * (345 * steps + 3500);
  const double k2 = q8_rounds(mid) * (570 * steps + 4500);
  // two a CU; the tiles past the last full round of them (see above)
  const double pair = 1050 * steps + 4000, one = 760 * steps + 4000, full = std::floor(mid / 512);
  const double k1 = mid <= 256 ? one
                    : mid <= 512 ? pair
                    : mid / 512 * pair + (mid > full * 512 ? (full < 2 ? 0.75 : 0.5) * one : 0);
  const double large = q8_rounds(q8_tiles(m, n, 128, 256)) * (1500 * steps + 5000);
  const double best = std::fmin(std::fmin(std::fmin(few, k3), std::fmin(k2, k1)), large);
  if (best == large) return {128, 256, 1};
  if (best == k1) return {64, 128, 1};
  if (best == k2) return {64, 128, 2};
  if (best == k3) return {32, 128, 3};
  return {64, 16, 1};
}

// bf16 activations: the kernel and tile that take the shortest time by these
// measured costs, linear in the 64-deep steps of k (ns; a round is 256 tiles,
// one for each CU, whether a CU holds one workgroup or several):
//   few rows   64 x 16    280 steps + 2000 a round
//   ring       32 x 128   400 steps + 400 a round + 2800
//              64 x 128   450 steps + 1000 a round + 3000
//             128 x 128   530 steps + 4000 for one round, else 610 steps + 2000 a round
//             160 x 128   660 steps + 5000 a round
//             128 x 256  1150 steps + 4000 a round
//             256 x 256  1600 steps + 5000 a round
// A lone small tile is bound by the latency of its serial k loop, and a 256 x
// 256 tile reads each operand least. One rule for all sizes instead of the
// first tile that covered every CU, us: 1029 x 1536 -> 9216 59 -> 46, 1536 x
// 2048 -> 8192 75 -> 59, 512 x 8192 -> 2048 70 -> 56, 512 x 1536 -> 1536 17 ->
// 13, 3000 x 1024 -> 3072 41 -> 31. Of 798 sizes timed with each tile (k 64 to
// 8192) the tile so chosen takes 1.0% longer than the shortest on average and
// 16% or less longer at all but those of 17 rows and 8192 columns (up to 36%)
// and 400 x 64 -> 9216 (24%). Groups of wavefronts that share k gain
// nothing here (512 x 8192 -> 2048: 61 us with four groups of 32 x 128): a
// workgroup of any tile already takes what one CU loads.
//
// Up to 16 rows as in f32 (us, few rows / 32 x 128: 16 x 4096 -> 32000 58 / 34,
// 1 x 4096 -> 32000 38 / 33, 16 x 1024 -> 16384 9.3 / 9.5, 8 x 1024 -> 24576
// 10.8 / 9.5, 1 x 1024 -> 24576 8.9 / 9.4, 16 x 1024 -> 8192 5.8 / 9.3).
inline Q8Tile q8_tile_bf16(int64_t m, int64_t n, int64_t k) {
  const double steps = (double)(k / 64);
  auto rounds = [&](int64_t bm, int64_t bn) { return q8_rounds(q8_tiles(m, n, bm, bn)); };
  if (m <= 16) {
    const double one_tile = q8_tiles(m, n, 16, 16) / 256 * steps * (68 + 2.75 * (double)m) + 2000;
    if (0.96 * one_tile <= rounds(32, 128) * 400 * steps + 3200) return {16, 16, 1};
    return {32, 128, 1};
  }
  const double r128 = rounds(128, 128);
  const Q8Tile tile[7] = {{64, 16, 1}, {32, 128, 1}, {64, 128, 1}, {128, 128, 1}, {160, 128, 1}, {128, 256, 1}, {256, 256, 1}};
  const double cost[7] = {m > kFewRowsMaxM ? INFINITY : rounds(64, 16) * (280 * steps + 2000),
                          rounds(32, 128) * (400 * steps + 400) + 2800,
                          rounds(64, 128) * (450 * steps + 1000) + 3000,
                          r128 == 1 ? 530 * steps + 4000 : r128 * (610 * steps + 2000),
                          rounds(160, 128) * (660 * steps + 5000),
                          rounds(128, 256) * (1150 * steps + 4000),
                          rounds(256, 256) * (1600 * steps + 5000)};
  int best = 6;  // the larger tile of two equal ones
  for (int i = 5; i >= 0; --i)
    if (cost[i] < cost[best]) best = i;
  return tile[best];
}

}  // namespace lux3d
