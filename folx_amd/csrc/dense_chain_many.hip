// A chain of narrow dense + activation layers (K, N <= 128) over many Jacobian rows, in four launches:
//   pack   the weights in the order in which the lanes take them, zeros past K and N
//   x      the values through all layers; f' and f'' of every layer stay in the workspace
//   rows   the Jacobian rows through all layers: z = row @ W, row <- f' z, and sum z^2 of a group of rows to the workspace
//   lap    the Laplacian through all layers: z = lap @ W, lap <- f' z + f'' sum z^2
//
// Layer by layer every Jacobian row goes to memory and back between two layers, which for layers this narrow takes as
// long as their products; here a row stays in the registers of one wavefront from the first layer to the last.  The product is
// formed transposed (v_mfma_f32_32x32x2_f32: D[column][position]), so that a lane holds, of position lane % 32, the columns
// 8 j + 4 (lane / 32) + i of the result -- which is just what it must supply as the second operand of the next layer's steps
// (j, i): no value crosses lanes, there is no LDS and no barrier.  Only the weights come from memory (L1 / L2), four steps
// to a 16-byte load, DEPTH loads ahead; f' and the sums of squares are laid out in the same order, one 16-byte access for four
// columns.  A column's products are added in the order of dense_act_kernel.
//
// What bounds it: at 100 features, 2000 positions and 400 rows (ten layers and a matrix-vector product) the rows take 1.48 ms, of
// which the matrix pipe is busy 83 % (128 columns formed for 100); the FP32 matrix instructions share their pipe with the other
// vector ones, some 160 a tile, so two wavefronts a SIMD would not hide them (and spill: 1.95 ms).  Rows per pass: T = 3 1.48 ms,
// T = 2 1.51 (the weights and f' serve more rows).  Left to the compiler, the loads sink to their use: 2.59 ms.  x and lap are one
// short chain each, 48 and 68 us.  us, layers one by one -> chain: the above 2047 -> 1612; the same over 800 positions 998 -> 787;
// six layers of 100, P = 40, 25 600 positions 1742 -> 1426; four of 52, P = 63, 5250: 197 -> 140; three of 20, P = 60, 20 000:
// 180 -> 121.  Fewer rows or layers lose to the x and lap passes (four of 100, P = 63, 100 positions: 137 -> 241) and inputs wider
// than 32 features to reading them across rows (two of 64 on 64 features, P = 48, 16 384: 202 -> 263, left to the layers).
#include "activations.h"
#include "dense_chain.h"

namespace {

using folx_chain::Layer;
using folx_chain::MAXL;
using folx_chain::Params;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int PB = 32;    // positions of a block: the columns of a 32 x 32 tile
constexpr int QF = 256;   // floats of one unit of operand order: 4 for each of 64 lanes
constexpr int DEPTH = 4;  // weights on their way

struct ManyParams {
  Params c;
  float *wp, *d1, *d2, *part;  // workspace
  int32_t n_layers;            // layers with a function
  int32_t G, PG;               // groups of Jacobian rows, rows of a group
  int64_t blocks;              // blocks of positions
};

template <int KS>
struct Shape {
  static constexpr int NT = (KS + 3) / 4;  // tiles of 32 columns
};

// ---------------------------------------------------------------------------------------------------------------- pack
// wp: layer 0 [NT][KS0][lane][4], the others [NT][KS][lane][4]; a matrix-vector product's [KS][lane][4]; DEPTH units of zeros
__global__ __launch_bounds__(64) void chain_pack_kernel(ManyParams a, int KS0, int KS, int units) {
  const int lane = threadIdx.x, lh = lane / 32, l32 = lane % 32;
  const int NT = (KS + 3) / 4;
  int u = blockIdx.x;
  const int first = NT * KS0, rest = NT * KS;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  int l, q, ks;
  if (u < first) { l = 0; q = u; ks = KS0; }
  else { l = 1 + (u - first) / rest; q = (u - first) % rest; ks = KS; }
  if (l < a.n_layers) {
    const Layer& ly = a.c.layer[l];
    const int col = 32 * (q / ks) + l32;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 8 * (q % ks) + 4 * lh + i;
      if (k < ly.K && col < ly.N) v[i] = ly.W[(int64_t)k * ly.N + col];
    }
  } else if (l < a.c.L && q < KS) {
    const Layer& ly = a.c.layer[l];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 8 * q + 4 * lh + i;
      if (k < ly.K) v[i] = ly.W[k];
    }
  }
  *reinterpret_cast<float4*>(a.wp + ((int64_t)u * 64 + lane) * 4) = make_float4(v[0], v[1], v[2], v[3]);
}

// four consecutive values of a row of N floats from column k on, zeros past its end
__device__ __forceinline__ floatx4 load4(const float* row, int k, int N, bool vec) {
  floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (vec) {
    if (k < N) v = *reinterpret_cast<const floatx4*>(row + k);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k + i < N) v[i] = row[k + i];
  }
  return v;
}
__device__ __forceinline__ void store4(float* row, int k, int N, bool vec, floatx4 v) {
  if (vec) {
    if (k < N) *reinterpret_cast<floatx4*>(row + k) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k + i < N) row[k + i] = v[i];
  }
}

// ------------------------------------------------------------------------------------------------------------ x and lap
// LDS traffic of this workgroup is complete; weights on their way stay on their way
__device__ __forceinline__ void line_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One workgroup for 32 positions, a wavefront for each tile of 32 columns; the operand goes through LDS, twice buffered.
template <int KS, bool LAP>
__global__ __launch_bounds__(64 * Shape<KS>::NT) void chain_line_kernel(ManyParams a, int KS0, bool vec_in) {
  constexpr int NT = Shape<KS>::NT, LD = 8 * KS + 4;
  __shared__ __attribute__((aligned(16))) float tile[2][PB * LD];
  const int lane = threadIdx.x % 64, mt = folx_wave_id(), lh = lane / 32, n = lane % 32;
  const int64_t b = blockIdx.x, r = b * PB + n;
  const bool live = r < a.c.R;
  const int64_t rc = live ? r : a.c.R - 1;
  const float* in = LAP ? a.c.lap : a.c.x;
  for (int q = mt; q < KS0; q += NT)
    *reinterpret_cast<floatx4*>(&tile[0][n * LD + 8 * q + 4 * lh]) = load4(in + rc * a.c.layer[0].K, 8 * q + 4 * lh, a.c.layer[0].K, vec_in);
  const float* w = a.wp + lane * 4;
  int ks = KS0, cur = 0;
  floatx4 wv[KS];
#pragma unroll
  for (int j = 0; j < KS; ++j)
    if (j < ks) wv[j] = *reinterpret_cast<const floatx4*>(w + (int64_t)(mt * ks + j) * QF);
  w += (int64_t)NT * ks * QF;
  __syncthreads();
  for (int l = 0; l < a.n_layers; ++l) {
    const Layer& ly = a.c.layer[l];
    const int64_t at = (((int64_t)l * a.blocks + b) * KS + 4 * mt) * QF + lane * 4;
    floatx4 d1[4], d2[4], sq[4];
    if constexpr (LAP) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * mt + j < KS) {
          d1[j] = *reinterpret_cast<const floatx4*>(a.d1 + at + j * QF);
          d2[j] = *reinterpret_cast<const floatx4*>(a.d2 + at + j * QF);
          sq[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      const float* part = a.part + (((int64_t)l * a.blocks + b) * a.G * KS + 4 * mt) * QF + lane * 4;
      int g = 0;
      for (; g + 4 <= a.G; g += 4) {  // four groups' sums on their way together, added in order
        floatx4 t[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (4 * mt + j < KS) t[u][j] = *reinterpret_cast<const floatx4*>(part + ((int64_t)(g + u) * KS + j) * QF);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (4 * mt + j < KS) sq[j] += t[u][j];
      }
      for (; g < a.G; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (4 * mt + j < KS) sq[j] += *reinterpret_cast<const floatx4*>(part + ((int64_t)g * KS + j) * QF);
    }
    floatx16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < KS; ++j)
      if (j < ks) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(&tile[cur][n * LD + 8 * j + 4 * lh]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[j][i], v[i], acc, 0, 0, 0);
      }
    if (l + 1 < a.n_layers) {  // the next layer's weights come while this one is finished
#pragma unroll
      for (int j = 0; j < KS; ++j) wv[j] = *reinterpret_cast<const floatx4*>(w + (int64_t)(mt * KS + j) * QF);
      w += (int64_t)NT * KS * QF;
    }
    float o[16];
    if constexpr (LAP) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (4 * mt + i / 4 < KS) o[i] = d1[i / 4][i % 4] * acc[i] + d2[i / 4][i % 4] * sq[i / 4][i % 4];
    } else {
      float f1[16], f2[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int col = 32 * mt + 8 * (i / 4) + 4 * lh + i % 4;
        acc[i] += ly.bias && col < ly.N ? ly.bias[col] : 0.0f;
      }
#define FOLX_CHAIN_CASE(A) \
  case A: _Pragma("unroll") for (int i = 0; i < 16; ++i) act_eval<A>(acc[i], ly.prm, o[i], f1[i], f2[i]); break;
      switch (ly.act) {
        FOLX_CHAIN_CASE(FOLX_ACT_TANH) FOLX_CHAIN_CASE(FOLX_ACT_SILU) FOLX_CHAIN_CASE(FOLX_ACT_LOGISTIC)
        FOLX_CHAIN_CASE(FOLX_ACT_SOFTPLUS) FOLX_CHAIN_CASE(FOLX_ACT_EXP) FOLX_CHAIN_CASE(FOLX_ACT_SIN)
        FOLX_CHAIN_CASE(FOLX_ACT_COS) FOLX_CHAIN_CASE(FOLX_ACT_GELU) FOLX_CHAIN_CASE(FOLX_ACT_GELU_TANH)
        default: _Pragma("unroll") for (int i = 0; i < 16; ++i) act_eval<FOLX_ACT_SQUARE>(acc[i], ly.prm, o[i], f1[i], f2[i]); break;
      }
#undef FOLX_CHAIN_CASE
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * mt + j < KS) {
          floatx4 f;
#pragma unroll
          for (int i = 0; i < 4; ++i) f[i] = 32 * mt + 8 * j + 4 * lh + i < ly.N ? f1[4 * j + i] : 0.0f;
          *reinterpret_cast<floatx4*>(a.d1 + at + j * QF) = f;
          *reinterpret_cast<floatx4*>(a.d2 + at + j * QF) = floatx4{f2[4 * j], f2[4 * j + 1], f2[4 * j + 2], f2[4 * j + 3]};
        }
    }
    const bool last = l + 1 == a.n_layers;
    float* out = a.c.L > a.n_layers ? (LAP ? a.c.h_lap : a.c.h) : (LAP ? a.c.y_lap : a.c.y);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * mt + j < KS) {
        const int k = 32 * mt + 8 * j + 4 * lh;
        floatx4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = k + i < ly.N ? o[4 * j + i] : 0.0f;
        if (last && out && live) store4(out + r * ly.N, k, ly.N, a.c.vec, v);
        *reinterpret_cast<floatx4*>(&tile[cur ^ 1][n * LD + k]) = v;
      }
    ks = KS;
    cur ^= 1;
    line_barrier();
  }
  if (a.c.L > a.n_layers && mt == 0) {
    float s = 0.0f;
    for (int j = 0; j < KS; ++j) {
      const floatx4 v = *reinterpret_cast<const floatx4*>(&tile[cur][n * LD + 8 * j + 4 * lh]);
      const floatx4 m = *reinterpret_cast<const floatx4*>(w + (int64_t)j * QF);
#pragma unroll
      for (int i = 0; i < 4; ++i) s = fmaf(v[i], m[i], s);
    }
    s += __shfl_xor(s, 32);
    const float* bias = a.c.layer[a.n_layers].bias;
    if (lh == 0 && live) (LAP ? a.c.y_lap : a.c.y)[r] = !LAP && bias ? s + bias[0] : s;
  }
}

// ----------------------------------------------------------------------------------------------------------------- rows
struct Line {
  floatx4 f[4], sq[4];  // f' and the sums so far of a tile's columns
};

template <int KS>
__device__ __forceinline__ void line_load(Line& v, const float* d1, const float* part, int mt) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (4 * mt + j < KS) {
      v.f[j] = *reinterpret_cast<const floatx4*>(d1 + (4 * mt + j) * QF);
      v.sq[j] = *reinterpret_cast<const floatx4*>(part + (4 * mt + j) * QF);
    }
}

// Columns 8 (4 mt + j) .. of a finished tile: the rows times f', their squares to the sums.
template <int KS, int T>
__device__ __forceinline__ void rows_finish(const floatx16 (&acc)[T], const Line& v, floatx4 (&out)[T][KS], float* part, int mt, int j,
                                            bool add) {
  floatx4 sq;
#pragma unroll
  for (int i = 0; i < 4; ++i) sq[i] = add ? v.sq[j][i] : 0.0f;
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float z = acc[t][4 * j + i];
      sq[i] += z * z;
      out[t][4 * mt + j][i] = v.f[j][i] * z;  // f' is 0 past the last column
    }
  *reinterpret_cast<floatx4*>(part + (4 * mt + j) * QF) = sq;
}

// One layer for T rows of the 32 positions: the operand `in` (KSI units of four columns), the result in `out` (KS units).  `w` walks
// the packed weights, `ring` holds the next DEPTH units of them.  A tile is finished among the products of the next one -- the last
// tile of a layer among those of the next layer, whose steps read it last: `acc` and `line` hand it over.
template <int KSI, int KS, int T, bool FIRST>
__device__ __forceinline__ void rows_layer(const float*& w, floatx4 (&ring)[DEPTH], floatx16 (&acc)[T], Line& line,
                                           floatx4 (&in)[T][KSI], floatx4 (&out)[T][KS], const float* d1, float* part,
                                           float* part_before, bool add) {
  constexpr int NT = Shape<KS>::NT;
#pragma unroll
  for (int mt = 0; mt < NT; ++mt) {
    Line now;
    line_load<KS>(now, d1, part, mt);
    floatx16 c[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) c[t][i] = 0.0f;
#pragma unroll
    for (int j = 0; j < KSI; ++j) {
      const int u = (mt * KSI + j) % DEPTH;
      const floatx4 wv = ring[u];
      ring[u] = *reinterpret_cast<const floatx4*>(w + (mt * KSI + j + DEPTH) * QF);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < T; ++t) c[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[i], in[t][j][i], c[t], 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (j == (q + 1 < KSI ? q + 1 : KSI - 1)) {
          if (mt > 0) {
            if (4 * (mt - 1) + q < KS) rows_finish<KS, T>(acc, line, out, part, mt - 1, q, add);
          } else if constexpr (!FIRST && NT > 1) {
            if (4 * (NT - 1) + q < KS) rows_finish<KSI, T>(acc, line, in, part_before, NT - 1, q, add);
          }
        }
      __builtin_amdgcn_sched_barrier(0);  // loads stay where they are asked for, DEPTH units ahead
    }
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = c[t];
    line = now;
  }
  if constexpr (NT == 1)
#pragma unroll
    for (int q = 0; q < 4; ++q) rows_finish<KS, T>(acc, line, out, part, 0, q, add);
  w += NT * KSI * QF;
  // the ring continues where this layer ended: unit (NT * KSI) of it is the next layer's unit 0
  if constexpr ((NT * KSI) % DEPTH != 0) {
    floatx4 t[DEPTH];
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) t[u] = ring[(u + NT * KSI) % DEPTH];
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) ring[u] = t[u];
  }
}

template <int KS0, int KS, int T>
__device__ __forceinline__ void rows_pass(const ManyParams& a, int64_t b, int64_t g, int p, bool add, bool vec_in, int lane) {
  const int lh = lane / 32, n = lane % 32;
  const int64_t r = b * PB + n;
  const bool live = r < a.c.R;
  const int64_t rc = live ? r : a.c.R - 1;
  const float* w = a.wp + lane * 4;
  floatx4 ring[DEPTH];
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) ring[u] = *reinterpret_cast<const floatx4*>(w + u * QF);
  floatx4 A[T][KS], B[T][KS];
  const float* d1 = a.d1 + b * KS * QF + lane * 4;
  float* part = a.part + (b * a.G + g) * KS * QF + lane * 4;
  const int64_t d1_step = a.blocks * KS * QF, part_step = a.blocks * a.G * KS * QF;
  constexpr int NT = Shape<KS>::NT;
  floatx16 acc[T];
  Line line;
  auto finish = [&](floatx4 (&out)[T][KS]) __attribute__((always_inline)) {
    if constexpr (NT > 1)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (4 * (NT - 1) + q < KS) rows_finish<KS, T>(acc, line, out, part, NT - 1, q, add);
  };
  {
    floatx4 in[T][KS0];
    const int K = a.c.layer[0].K;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < KS0; ++j) in[t][j] = load4(a.c.jac + ((int64_t)(p + t) * a.c.R + rc) * K, 8 * j + 4 * lh, K, vec_in);
    rows_layer<KS0, KS, T, true>(w, ring, acc, line, in, A, d1, part, part, add);
  }
  int l = 1;
  for (; l + 1 < a.n_layers; l += 2) {
    d1 += d1_step;
    part += part_step;
    rows_layer<KS, KS, T, false>(w, ring, acc, line, A, B, d1, part, part - part_step, add);
    d1 += d1_step;
    part += part_step;
    rows_layer<KS, KS, T, false>(w, ring, acc, line, B, A, d1, part, part - part_step, add);
  }
  if (l < a.n_layers) {
    d1 += d1_step;
    part += part_step;
    rows_layer<KS, KS, T, false>(w, ring, acc, line, A, B, d1, part, part - part_step, add);
    finish(B);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < KS; ++j) A[t][j] = B[t][j];
  } else {
    finish(A);
  }
  const bool vector = a.c.L > a.n_layers;
  float* out = vector ? a.c.h_jac : a.c.y_jac;
  const int N = a.c.layer[a.n_layers - 1].N;
  if (out && live)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float* row = out + ((int64_t)(p + t) * a.c.R + r) * N;
#pragma unroll
      for (int j = 0; j < KS; ++j) store4(row, 8 * j + 4 * lh, N, a.c.vec, A[t][j]);
    }
  if (vector) {
    float s[T];
#pragma unroll
    for (int t = 0; t < T; ++t) s[t] = 0.0f;
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      const floatx4 m = *reinterpret_cast<const floatx4*>(w + j * QF);
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[t] = fmaf(A[t][j][i], m[i], s[t]);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      s[t] += __shfl_xor(s[t], 32);
      if (lh == 0 && live) a.c.y_jac[(int64_t)(p + t) * a.c.R + r] = s[t];
    }
  }
}

// A wavefront owns one group of Jacobian rows of one block of positions, T rows at a time, what is left one by one.
template <int KS0, int KS, int T>
__global__ __launch_bounds__(256, 1) void chain_rows_kernel(ManyParams a, bool vec_in) {
  const int lane = threadIdx.x % 64;
  const int64_t u = (int64_t)blockIdx.x * 4 + folx_wave_id();
  if (u >= a.blocks * a.G) return;
  const int64_t b = u / a.G;
  const int g = (int)(u - b * a.G);
  int p = g * a.PG;
  const int p0 = p, p1 = min(a.c.P, p + a.PG);
  for (; p + T <= p1; p += T) rows_pass<KS0, KS, T>(a, b, g, p, p > p0, vec_in, lane);
  for (; p < p1; ++p) rows_pass<KS0, KS, 1>(a, b, g, p, p > p0, vec_in, lane);
}

struct Plan {
  int ks0, ks, nt, units;
  bool faster;
  int32_t n_layers, G, PG;
  int64_t blocks, line_floats, part_floats;  // floats of f' / f'' / of the sums of squares
};

constexpr int64_t SIMDS = 1024;

bool plan_many(int L, const int32_t* act, const int32_t* widths, int64_t R, int32_t P, Plan& pl) {
  if (L < 1 || L > MAXL || P < 1) return false;
  const bool vector = act[L - 1] < 0;
  if (vector && widths[L] != 1) return false;
  pl.n_layers = L - vector;
  if (pl.n_layers < 1 || widths[0] > 32) return false;
  int widest = 0;
  for (int l = 0; l <= pl.n_layers; ++l) {
    if (widths[l] < 1 || widths[l] > 128) return false;
    if (l > 0 && widths[l] > widest) widest = widths[l];
  }
  for (int l = 0; l < pl.n_layers; ++l)
    switch (act[l]) {
      case FOLX_ACT_TANH: case FOLX_ACT_SILU: case FOLX_ACT_LOGISTIC: case FOLX_ACT_SOFTPLUS: case FOLX_ACT_EXP:
      case FOLX_ACT_SIN: case FOLX_ACT_COS: case FOLX_ACT_SQUARE: case FOLX_ACT_GELU: case FOLX_ACT_GELU_TANH: break;
      default: return false;
    }
  pl.ks = widest <= 32 ? 4 : (widest <= 64 ? 8 : (widest <= 104 ? 13 : 16));
  pl.ks0 = widths[0] <= 8 ? 1 : 4;
  pl.nt = (pl.ks + 3) / 4;
  pl.units = pl.nt * (pl.ks0 + (pl.n_layers - 1) * pl.ks) + pl.ks + DEPTH;
  pl.blocks = (R + PB - 1) / PB;
  // as many groups of rows as keep the wavefronts' shares equal on the chip's SIMDs, at least eight rows each
  int64_t best = 0;
  pl.G = 1;
  for (int32_t G = 1; G <= (P > 8 ? P / 8 : 1) && (G == 1 || pl.blocks * G <= 4 * SIMDS); ++G) {
    const int64_t PG = (P + G - 1) / G;
    const int64_t cost = ((pl.blocks * G + SIMDS - 1) / SIMDS) * PG;
    if (best == 0 || cost < best) { best = cost; pl.G = G; }
  }
  pl.PG = (P + pl.G - 1) / pl.G;
  pl.G = (P + pl.PG - 1) / pl.PG;
  pl.line_floats = pl.n_layers * pl.blocks * pl.ks * QF;
  pl.part_floats = pl.line_floats * pl.G;
  // Microseconds of the chain: the matrix pipe at 2.35 GHz, 85 % of it busy, in the layers' share of the busiest SIMD, a
  // line kernel's layer, launches -- and of the layers one by one: 80 % of the sum of their traffic at 5.3 TB/s and
  // their products (neither hides all of the other), launches.  Within 30 % of both sides at the sizes above; the layers are
  // taken too cheap below 1000 positions, where the two sides are close.
  const double cycles = 256.0 * pl.nt;  // of a unit of a layer's operand: 4 steps of 64 cycles for every tile
  const double rounds = (double)((pl.blocks * pl.G + SIMDS - 1) / SIMDS);
  double chain = 15.0 + rounds * pl.PG * (pl.ks0 + (pl.n_layers - 1.0) * pl.ks) * cycles / (2350.0 * 0.85) +
                 pl.n_layers * (4.0 + 0.6 * pl.ks) * (double)((pl.blocks + 511) / 512);
  double layers = 0.0;
  for (int l = 0; l < L; ++l) {
    const double K = widths[l], N = widths[l + 1], ks = K <= 8 ? 1 : (K <= 32 ? 4 : (K <= 64 ? 8 : (K <= 104 ? 13 : 16)));
    const double nt = N <= 32 ? 1 : (N <= 64 ? 2 : 4);
    const double bytes = 4.0 * (P + 2) * R * (K + N), mem = bytes / 5.3e6;
    const double mfma = l < pl.n_layers ? (P + 2.0) * pl.blocks * nt * ks * 256.0 / (SIMDS * 2350.0) : 0.0;
    layers += 0.8 * (mem + mfma) + (pl.blocks < 384 ? 12.0 : 5.0);
  }
  pl.faster = chain < layers;
  return pl.blocks * pl.G <= 0x7fffffffLL;
}

template <int KS0, int KS, int T>
int launch(hipStream_t st, const ManyParams& a, const Plan& pl, bool vec_x, bool vec_j, bool vec_l) {
  constexpr int NT = Shape<KS>::NT;
  chain_pack_kernel<<<dim3((unsigned)pl.units), dim3(64), 0, st>>>(a, KS0, KS, pl.units);
  chain_line_kernel<KS, false><<<dim3((unsigned)a.blocks), dim3(64 * NT), 0, st>>>(a, KS0, vec_x);
  chain_rows_kernel<KS0, KS, T><<<dim3((unsigned)((a.blocks * a.G + 3) / 4)), dim3(256), 0, st>>>(a, vec_j);
  chain_line_kernel<KS, true><<<dim3((unsigned)a.blocks), dim3(64 * NT), 0, st>>>(a, KS0, vec_l);
  return folx_launch_status();
}

}  // namespace

namespace folx_chain {

bool many_plan(int L, const int32_t* act, const int32_t* widths, int64_t R, int32_t P, bool& faster, int64_t& ws_bytes) {
  Plan pl;
  if (!plan_many(L, act, widths, R, P, pl)) return false;
  ws_bytes = ((int64_t)pl.units * QF + 2 * pl.line_floats + pl.part_floats) * 4;
  faster = pl.faster;
  return true;
}

int many_launch(hipStream_t st, const Params& c, const int32_t* act, const int32_t* widths, void* ws) {
  Plan pl;
  if (!plan_many(c.L, act, widths, c.R, c.P, pl)) return FOLX_HIP_ENOTSUP;
  ManyParams a;
  a.c = c;
  a.n_layers = pl.n_layers;
  a.G = pl.G;
  a.PG = pl.PG;
  a.blocks = pl.blocks;
  a.wp = (float*)ws;
  a.d1 = a.wp + (int64_t)pl.units * QF;
  a.d2 = a.d1 + pl.line_floats;
  a.part = a.d2 + pl.line_floats;
  const bool k4 = widths[0] % 4 == 0;
  const bool vx = k4 && folx_aligned16(c.x), vj = k4 && folx_aligned16(c.jac), vl = k4 && folx_aligned16(c.lap);
  if (pl.ks0 == 1) switch (pl.ks) {
      case 4: return launch<1, 4, 8>(st, a, pl, vx, vj, vl);
      case 8: return launch<1, 8, 4>(st, a, pl, vx, vj, vl);
      case 13: return launch<1, 13, 3>(st, a, pl, vx, vj, vl);
      default: return launch<1, 16, 2>(st, a, pl, vx, vj, vl);
    }
  switch (pl.ks) {
    case 4: return launch<4, 4, 8>(st, a, pl, vx, vj, vl);
    case 8: return launch<4, 8, 4>(st, a, pl, vx, vj, vl);
    case 13: return launch<4, 13, 3>(st, a, pl, vx, vj, vl);
    default: return launch<4, 16, 2>(st, a, pl, vx, vj, vl);
  }
}

}  // namespace folx_chain
