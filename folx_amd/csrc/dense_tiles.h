// Which tiles a plain product takes, and the matrix work that follows: host code shared by the dense rule and by the plan of
// the wide fused rule, which has to know what the product that it would replace costs.
#pragma once
#include <stdint.h>

// Time of a product of `rows` (three segments) with N > 64 columns, in 64 x 64 tiles per CU and feature; `small`: whether
// 64 x 64 tiles are the faster ones.
// A CU works through its share of 128 x 256 tiles (8 units of 64 x 64; 128 x 128: 4) at the rate of the matrix pipe,
// however many share it, so a launch takes ceil(tiles / 256) tile times; 64 x 64 tiles divide finer, also the columns
// (N = 160 is 192 instead of 256), at an eighth less rate (twice the LDS reads per product).  us, large -> small:
// K = N = 256: 1280 rows 36 -> 10, 20 480 (160 tiles) 40 -> 30, 47 104 (368) 73 -> 62, 82 432 (644) 105 -> 101; 159 900 rows
// (1249 tiles) would go 173 -> 191.  K = N = 128: 9984 rows 14.1 -> 8.6, 69 984 33.5 -> 28.5, 140 000 55.9 -> 50.2; 300 000 would
// go 98.8 -> 100.1.  K = 512, N = 100: 140 000 rows 180 -> 174, 300 000 would go 351 -> 364; K = 64: 66 -> 62 there, which
// the rule leaves.  Over 196 sizes (N = 68 .. 512, K = 16 .. 512, 1000 .. 300 000 rows) its choice was slower than the large tiles once, by
// 6 % (N = 132, K = 16, 140 000 rows).  The opt-in products have the 128 x 256 tile only.
inline double folx_dense_units(const int64_t (&rows)[3], int32_t N, bool split, bool& small) {
  int64_t nb = 0, ns = 0;
  for (int64_t r : rows) { nb += (r + 127) / 128; ns += (r + 63) / 64; }
  nb *= N > 128 ? (N + 255) / 256 : 1;
  ns *= (N + 63) / 64;
  const double big = (N > 128 ? 8.0 : 4.0) * (double)((nb + 255) / 256), fine = 1.16 * (double)ns / 256;
  small = (N <= 128 || !split) && fine < big;
  return small ? fine : big;
}
