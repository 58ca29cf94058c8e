// What products of rows are expected to take on the tiles they may have, where that is a matter of counting: host code alone.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace ughip {

// What a product of rows takes at most of the device's block, which stays as large as the largest call made it, where it can do without: 128 MiB are the sums of 2978 rows of 2 x 5632, and of a product with more the tiles
// of 32 to 128 rows would gain 9 % at most (6144 rows of 5632 x 2048 1185 us for 1300 by the prices, 16384 of 2 x 5632 4 %, with 738 MB).
constexpr size_t ROWS_BLOCK_MOST = (size_t)128 << 20;

// How rows by group are spread is not known where a product is planned: a router's experts come out with shares that differ by 40 % or so, the share of an even one's rows times one of these for a sixteenth of the groups each.
constexpr double SHARES[16] = {.44, .55, .62, .68, .73, .79, .84, .90, .95, 1.02, 1.08, 1.16, 1.26, 1.38, 1.56, 1.94};
inline int share_rows(int m, int groups, double share) { return std::max(1, (int)((double)m / groups * share + 0.999)); }
// how many tiles of bm rows m rows by group are expected to be, as the f32 prices below were fitted to it: by eighths
inline double grouped_tile_rows(int m, int groups, int bm) {
  double n = 0;
  for (double share : {0.50, 0.65, 0.76, 0.87, 0.98, 1.12, 1.32, 1.70}) n += groups / 8.0 * ((share_rows(m, groups, share) + bm - 1) / bm);
  return n;
}

// f32 (rows_product): which of 128 x 128, 64 x 128 and 64 x 64 (22, 12, 11).  An f32 MFMA has its SIMD to itself, so a second tile on a CU takes as long again: a product lasts for as many rounds of 256 tiles
// as it has, whole ones and one at least, at what a tile takes by itself (us per 2048 of K), and the larger tile's better rate is often less than the smaller one's fuller last round.  us on 22 / 12 / 11: gated
// n 5632, k 2048, 100 rows 152 / 91, 300 rows 285 / 172, 509 296 / 258, 700 430 / 336, 1024 448 / 486; n 10304, k 2048, 509 rows 296 / 254 / 266; n 6592, 700 rows 290 / 246 / 231; n 2048,
// 1531 rows 163 / 164 / 148; gated n 2816, k 1024, 300 rows 84 / 51, 700 151 / 91; 16 groups, gated n 1408, 1200 rows 296 / 251, 2036 rows 318 / 334.
inline int f32_rows_tile(int m, int n, int k, int groups, bool gated, double* price_us = nullptr) {
  int best = 0;
  double best_us = 0;
  for (int tile : {22, 12, 11}) {
    if (gated && tile == 11) continue;  // a tile's columns come in gate / up pairs
    const int bm = tile == 22 ? 128 : 64, cols = (tile == 11 ? 64 : 128) / (gated ? 2 : 1);
    if (best && (m + bm - 1) / bm + groups > 65535) continue;  // tile rows are a grid's second dimension
    // (by group a few tiles more than expected may be a round: 1200 rows on 128 x 128, n 2048 of k 1408, 201 us where 16 tile rows would be 108, 64 x 128 124)
    const double rows = groups > 1 ? 1.06 * grouped_tile_rows(m, groups, bm) : (m + bm - 1) / bm, tiles = rows * ((n + cols - 1) / cols);
    const double rounds = std::max(1.0, std::ceil(tiles / 256 - (groups > 1 ? 0.01 : 0.0)));
    const double us = 4.0 + rounds * k / 2048.0 * (tile == 22 ? 144.0 : tile == 12 ? 81.0 : 45.5);
    if (!best || us < best_us * 0.97) best = tile, best_us = us;
  }
  if (price_us) *price_us = best_us;
  return best;
}

// The tile of what is not gated where f32_rows_tile does not choose it, in bf16 and with a lookup.  rows: of a group, or m
inline int rows_tile(int m, int n, int rows) { return rows > 64 && (long long)((m + 127) / 128) * ((n + 127) / 128) >= 192 ? 22 : 11; }
// f32 products with a lookup on that tile: what a product without one takes there, and the table's scattered elements, by rounds of the large tile (us, k 128: 1024 rows of n 5632 50, 2000 75; 100 of n 64, k 512 17.1, without a lookup 14.6)
inline double f32_lookup_us(int m, int n, int k) {
  const int tile = rows_tile(m, n, m), t = tile == 22 ? 128 : 64;
  const double rounds = std::max(1.0, std::ceil((double)((m + t - 1) / t) * ((n + t - 1) / t) / 256));
  return 4.0 + rounds * k / 2048.0 * (tile == 22 ? 144.0 : 45.5) + (tile == 22 ? 14.0 * rounds : 2.5);
}

// f32 rows against an f32 matrix: gemm_tiled's tiles, at their price (negative: they do not take it) and with `bytes` for what lies between them and the fold, or rows_product's.  2 us are the tiles' longer way in.
inline bool f32_rows_on_tiles(double tiles_us, double rows_product_us, size_t bytes) { return tiles_us >= 0 && tiles_us + 2.0 < 0.97 * rows_product_us && bytes <= ROWS_BLOCK_MOST; }

// bf16 products of f32 rows: rows_product, which rounds on its way to LDS and has one chain of steps, or a launch that rounds the rows ahead (k % 64 == 0) and the tiles of bf16 rows, two launches of 5.7 us before
// anything else.  What either takes, us: fitted to 2500 products whose matrices come from caches and 240 from memory (2 to 3000 rows; plain, gated, with a lookup, 2 to 64 groups; n 32 to 6000, k 64 to 5632), 13 and 10 % off
// in the mean square.
inline double rounded_on_the_way_us(int m, int n, int k, int groups, bool gated, bool lookup) {
  const int rows = groups ? (m + groups - 1) / groups : m, met = groups ? std::min(groups, m) : 1;  // matrices that rows meet
  const int tile = gated ? (rows > 64 ? 22 : 12) : rows_tile(m, n, rows), bm = tile == 22 ? 128 : 64, cols = (tile == 11 ? 64 : 128) / (gated ? 2 : 1);
  static const struct {
    double fixed, height, step, past_step, past, mb;  // height: of a tile's, that rows fill; past: for every round of 256 tiles behind the first; mb: of the matrices
  } prices[] = {{2.89, 1.39, 0.775, 0.629, 1.9, 0.0}, {2.37, 2.67, 0.578, 0.168, 1.1, 0.059}, {5.69, 0.99, 0.917, 0.706, 3.2, 0.012}};
  const auto& p = prices[tile == 11 ? 0 : tile == 12 ? 1 : 2];
  const double high = (double)std::min(rows, bm) / bm, past = std::max(0.0, (double)met * ((rows + bm - 1) / bm) * ((n + cols - 1) / cols) / 256 - 1);
  const int steps = tile == 11 ? (k + 127) / 128 : (k + 63) / 64;
  // (a lookup's rows of the table are scattered: 128 x 128 of its elements are asked for by each tile)
  return p.fixed + p.height * high + steps * (p.step + p.past_step * past) + p.past * past + p.mb * 2e-6 * met * (gated ? 2.0 : 1.0) * n * k + 0.095 * groups +
         (!lookup ? 0 : tile == 22 ? 23.0 : 1.47 + 1.18 * high);
}
inline double rounded_ahead_us(int m, int n, int k, int groups, bool gated) {
  const int rows = groups ? (m + groups - 1) / groups : m, met = groups ? std::min(groups, m) : 1;
  const double columns = (gated ? 2.0 : 1.0) * n, past = std::max(0.0, (double)met * ((rows + 127) / 128) * std::ceil(columns / 128) / 256 - 1);  // as tiles of 128 x 128
  const double us = 5.69 + k / 64 * (0.086 + 0.159 * past) + 1.15 * past + 0.106e-6 * (2.0 * met * columns * k) + 0.169e-6 * (6.0 * m * k) + 0.184e-6 * (4.0 * m * n) + 0.65e-9 * (m * columns * k);
  return std::max(5.8, us);
}
// Ahead where it is clearly the faster one: of the products from caches 1.1 % from the faster one in the mean, 7 of them 4 % and more (13 % at most) slower than on the way; from memory 1.9 %, none.  us on the way / ahead: gated, 2
// rows, n 64, k 64 3.3 / 6.2, k 512 6.8 / 5.9, k 2048 19.9 / 9.3; 130 rows, k 64 6.7 / 5.9; lookups, 2 rows, n 704, k 128 5.0 / 6.0, k 512 7.2 / 5.9; 4 groups, 32 rows, n 704, k 128 4.3 / 6.4, k 1024 9.1 / 8.2; 64 groups, 64
// rows, n 64, k 64 9.6 / 6.0; 16 groups, 64 rows, gated, k 1024, n 704 17.2 / 12.9, n 1408 20.8 / 18.8, n 2048 22.7 / 26.9; plain with a bias, n 2048, 16 rows k 384 5.7 / 6.0, k 768 7.7 / 6.9, k 1024 9.1 / 6.7, 300 rows k
// 640 8.0 / 8.8.
inline bool rows_rounded_ahead(int m, int n, int k, int groups, bool gated, bool lookup) {
  return rounded_on_the_way_us(m, n, k, groups, gated, lookup) > 1.06 * rounded_ahead_us(m, n, k, groups, gated);
}

// How many of a head's vdim results a workgroup of latent_merge makes, of 16, 32, 64 and 128 (latent_attention.hip): every one adds all parts of its row up, so as few workgroups to a row as leave no CU idle, the least number of
// results that is one round of them, and no more than there are.  us for all three launches on 16 / 32 / 64 / 128, f32, rank 512: vdim 128, 64 rows 18.4 / 16.1 / 16.7 / 19.0, 96 21.2 / 19.2 / 17.2 / 19.4, 128 24.2 / 20.0 / 18.1 /
// 20.5, 256 35.2 / 27.3 / 23.5 / 22.4, 2048 192 / 128 / 97 / 87; vdim 64, 128 rows 19.3 / 17.1 / 17.6 / 18.6, 192 22.9 / 20.8 / 18.8 / 19.7; vdim 16, 1024 rows 37.0 / 37.1 / 37.7 / 40.3.
inline int latent_merge_results(size_t rows, size_t vdim, int cus) {
  int v = 16;
  while (v < 128 && (size_t)v < vdim && rows * ((vdim + v - 1) / v) > (size_t)cus) v *= 2;
  return v;
}

}  // namespace ughip
