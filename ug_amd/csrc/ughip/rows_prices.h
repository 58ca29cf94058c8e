// What products of rows are expected to take on the tiles they may have, where that is a matter of counting: host code alone.
#pragma once
#include <algorithm>
#include <cmath>

namespace ughip {

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

}  // namespace ughip
