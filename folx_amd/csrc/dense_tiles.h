// Which tiles a plain product takes, and the matrix work that follows: host code shared by the dense rule and by the plan of
// the wide fused rule, which has to know what the product that it would replace costs.
#pragma once
#include <hip/hip_runtime.h>
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

// What a launch of the products from bf16 pieces (SplitTile) takes, in us: the launch and the chain of its first tile, the work
// of a CU that holds all the workgroups it can per contracted feature and around the loop, and a MB of traffic beside it; `alone`
// is the share of that work's time which one workgroup on a CU takes.  Fitted to 520 products (R = 200 .. 48 000, P = 2 .. 120,
// K = 16 .. 512, N = 132 .. 512, every form of each timed): 8 to 12 % rms.
struct PiecesRates {
  int blocks, slots;  // blocks of 32 columns of a tile, workgroups on a CU
  double launch, chain, feature, around, mb, alone;
};

inline double folx_pieces_time(const PiecesRates& c, int64_t workgroups, int32_t K, double mb) {
  const int64_t room = 256 * c.slots, rest = workgroups % room;
  double units = (double)(workgroups / room);
  if (rest > 0) {
    const int64_t most = (rest + 255) / 256;  // on the fullest CU
    units += c.alone + (1.0 - c.alone) * (double)(most - 1) / (c.slots - 1);
  }
  return c.launch + c.chain * K + units * (c.feature * K + c.around) + c.mb * mb;
}

// The plain rule: 8 blocks with W prepared by a launch of its own, 4 and 2 with W split by every workgroup.
constexpr PiecesRates PIECES_PLAIN[3] = {{8, 2, 24.9, 0.0, 0.0953, 1.34, 0.109, 0.61},
                                         {4, 3, 13.6, 0.0, 0.1087, 3.44, 0.038, 0.38},
                                         {2, 4, 10.3, 0.0, 0.0917, 3.91, 0.002, 0.27}};

// The blocks of a tile with the least estimated time (8, 4 or 2; all add in the same order), and that time.  Of the 520 products it
// takes 1.016 times the fastest form's time in the mean; the most blocks that still give every CU a workgroup: 1.096.
inline int folx_pieces_columns(const int64_t (&rows)[3], int32_t K, int32_t N, double* time = nullptr) {
  int64_t tiles = 0, total = 0;
  for (int64_t r : rows) { tiles += (r + 127) / 128; total += r; }
  int best = 0;
  double least = 0.0;
  for (const PiecesRates& c : PIECES_PLAIN) {
    const double t = folx_pieces_time(c, tiles * ((N + 32 * c.blocks - 1) / (32 * c.blocks)), K, 4e-6 * (double)total * (K + N));
    if (best == 0 || t < least) { best = c.blocks; least = t; }
  }
  if (time != nullptr) *time = least;
  return best;
}

// Value and Laplacian rows of the dense rule from bf16 pieces (K a multiple of 16, x and lap 16-byte aligned).  pieces:
// folx_split::pieces_bytes of memory; with W given its pieces are formed there on the way, without it they are there already.
int folx_dense_values(hipStream_t st, const float* x, const float* lap, const float* W, char* pieces, const float* bias, float* y,
                      float* y_lap, int64_t R, int32_t K, int32_t N);
