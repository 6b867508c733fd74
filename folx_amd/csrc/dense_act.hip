// Narrow dense layer and its activation in one pass:
//   z = x @ W + bias          y     = f(z)
//   zj[p] = jac[p] @ W        yj[p] = f'(z) * zj[p]
//   zl = lap @ W              yl    = f'(z) * zl + f''(z) * sum_p zj[p]^2
// for K, N <= 128.  The pre-activation triplet never goes to HBM: the layer reads its input
// triplet once and writes its output triplet once, which is what bounds a layer this narrow.
//
// A workgroup of 4 wavefronts owns BR consecutive rows (positions) and ALL N columns, and walks
// the operand one Jacobian row at a time: x first (which gives f' and f'' for its rows, kept
// in registers), then its Jacobian rows (scaled by f' on the way out, squares summed in
// registers), then lap.  The BR x K input tile of one step is contiguous in memory and goes
// straight into LDS (global_load_lds_dwordx4), double buffered.  W never touches LDS: each
// wavefront owns a strip of 32 columns and keeps its K x 32 slice of W in registers as
// ready-made MFMA operands (v_mfma_f32_32x32x2_f32; lane l, register (j, i) <-> k = 8 j +
// 4 (l / 32) + i, column l % 32, matching the 128-bit reads of the A tile).
//
// LDS layout of the tile: [row][K / 4 pieces of 16 bytes]; piece c of row m sits at slot
// c ^ rot(m), with rot chosen from the power of two in K / 4 so that 16 consecutive rows reading
// the same k land on different banks (no rotation when K / 4 is odd, e.g. K = 100).
//
// When there are few row tiles (a small batch) the Jacobian rows are split over G workgroups
// per row tile in a first launch, each of which leaves its partial sums of squares in the
// workspace; a second, short launch with one workgroup per row tile recomputes f' and f''
// from the x tile, adds the partials in a fixed order and produces the lap row.
#include <type_traits>

#include "activations.h"
#include "dense_act_wide.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) char gchar;    // global memory, so that stores stay global_store
typedef __attribute__((address_space(1))) float gfloat;

#define FOLX_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define FOLX_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

constexpr int NTHR = 256;
constexpr int TM = 1;                 // 32-row accumulator tiles per wavefront
constexpr int TILE_FLOATS = 4096;     // one LDS buffer
constexpr int MAXLD = TILE_FLOATS / 4 / NTHR;
constexpr int PART_PER_BLOCK = TM * 16 * NTHR;

struct DAParams {
  const float *x, *jac, *lap, *W, *bias;
  const float *res, *res_jac, *res_lap;  // optional triplet of the output's shape added to the activated result
  float *y, *y_jac, *y_lap;
  float* part;
  int64_t R;
  int32_t P, K, N, G, PG, act, mode;  // mode 0: whole rule, 1: x + Jacobian rows of one group, 2: lap from partials
  float prm;
};

struct DAPlan {
  int wc, ks, br;
  int64_t row_tiles;
  int32_t G, PG;
  int64_t ws_bytes;
};

// Returns false when the shape is outside what the kernel is built for.
bool plan_dense_act(int64_t R, int32_t P, int32_t K, int32_t N, DAPlan& pl) {
  if (K < 4 || K > 128 || K % 4 != 0 || N < 1 || N > 128) return false;
  pl.wc = (N <= 32 && K <= 32) ? 1 : ((N <= 64 && K <= 64) ? 2 : 4);
  pl.ks = K <= 8 ? 1 : (K <= 32 ? 4 : (K <= 64 ? 8 : (K <= 104 ? 13 : 16)));
  pl.br = 32 * TM * (4 / pl.wc);
  pl.row_tiles = (R + pl.br - 1) / pl.br;
  int64_t G = 1;
  if (pl.row_tiles > 0 && pl.row_tiles < 384) {
    G = 512 / pl.row_tiles;
    int64_t gmax = P / 8;
    if (G > gmax) G = gmax;
    if (G < 1) G = 1;
  }
  pl.G = (int32_t)G;
  pl.PG = (int32_t)((P + G - 1) / G);
  pl.G = pl.PG > 0 ? (P + pl.PG - 1) / pl.PG : 1;  // no empty group
  if (pl.row_tiles * pl.G > 0x7fffffffLL) return false;
  pl.ws_bytes = pl.G > 1 ? pl.row_tiles * pl.G * (int64_t)PART_PER_BLOCK * 4 : 0;
  return true;
}

template <int KS, int WC>
__global__ __launch_bounds__(NTHR, 2) void dense_act_kernel(DAParams a) {
  constexpr int WR = 4 / WC;
  constexpr int BR = 32 * TM * WR;
  __shared__ __attribute__((aligned(16))) float As0[TILE_FLOATS];
  __shared__ __attribute__((aligned(16))) float As1[TILE_FLOATS];

  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32;
  const int lh = lane / 32;
  const int wrow = (wave / WC) * 32 * TM;
  const int wcol = (wave % WC) * 32;
  const int K = a.K, N = a.N, G = a.G;
  const int npr = K / 4;
  const int64_t R = a.R;
  const int mode = a.mode;
  const int64_t rt = mode == 1 ? blockIdx.x / G : blockIdx.x;
  const int g = mode == 1 ? (int)(blockIdx.x % G) : 0;
  const int64_t r0 = rt * BR;
  const int p0 = g * a.PG;
  const int p1 = mode == 1 ? min(a.P, p0 + a.PG) : a.P;
  const int nJ = mode == 2 ? 0 : p1 - p0;
  const int n_iter = 1 + nJ + (mode != 1 ? 1 : 0);

  // bank rotation of the tile rows
  int sh = __builtin_ctz(npr);
  if (sh > 4) sh = 4;
  const int rshift = 4 - sh;
  const int rmask = (1 << sh) - 1;
  const int sw = (l32 >> rshift) & rmask;

  // which 16 bytes of the tile each lane asks for; lane i of a load lands at slot (wave base + i)
  const int pieces = BR * npr;  // a multiple of 64
  int32_t src_off[MAXLD];
#pragma unroll
  for (int i = 0; i < MAXLD; ++i) {
    const int q = i * NTHR + tid;
    int off = 0;
    if (q < pieces) {
      int m = q / npr;
      const int c = (q - m * npr) ^ ((m >> rshift) & rmask);
      if (r0 + m >= R) m = (int)(R - 1 - r0);
      off = m * K + 4 * c;
    }
    src_off[i] = off;
  }
  auto tile_src = [&](int it) __attribute__((always_inline)) -> const float* {
    if (it == 0) return a.x + r0 * K;
    if (it <= nJ) return a.jac + ((int64_t)(p0 + it - 1) * R + r0) * K;
    return a.lap + r0 * K;
  };
  auto issue = [&](const float* src, float* buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MAXLD; ++i)
      if (i * NTHR + wave * 64 < pieces)
        __builtin_amdgcn_global_load_lds(FOLX_GPTR(src + src_off[i]), FOLX_LPTR(&buf[(i * NTHR + wave * 64) * 4]),
                                         16, 0, 0);
  };

  // this wavefront's slice of W as MFMA operands
  const int col = wcol + l32;
  const bool col_ok = col < N;
  float wreg[KS][4];
#pragma unroll
  for (int j = 0; j < KS; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 8 * j + 4 * lh + i;
      wreg[j][i] = (k < K && col_ok) ? a.W[(int64_t)k * N + col] : 0.0f;
    }
  const float bcol = (a.bias != nullptr && col_ok) ? a.bias[col] : 0.0f;

  const int arow0 = (wrow + l32) * K;
  auto compute = [&](const float* buf, floatx16 (&acc)[TM]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
    // Every group of 8 k is multiplied, also past K: a lane whose 4 k lie past K reads the last
    // 4 k of its own row instead and meets zeros in the W registers, so the product is one
    // straight run of LDS reads and MFMAs with no test on the data, and no row ever sees
    // another row's values.  The reads run one group ahead of the MFMAs.
    auto frag = [&](int j, float4 (&av)[TM]) __attribute__((always_inline)) {
      const int ch = min(2 * j + lh, npr - 1);
#pragma unroll
      for (int t = 0; t < TM; ++t)
        av[t] = *reinterpret_cast<const float4*>(&buf[arow0 + t * 32 * K + ((ch ^ sw) * 4)]);
    };
    float4 av[2][TM];
    frag(0, av[0]);
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      if (j + 1 < KS) frag(j + 1, av[(j + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < TM; ++t) {
          const float4& q = av[j & 1][t];
          const float v = i == 0 ? q.x : (i == 1 ? q.y : (i == 2 ? q.z : q.w));
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, wreg[j][i], acc[t], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Register r of a 32x32 accumulator tile holds row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32.
  // The rows are stored in increasing order through one running row pointer: its steps are
  // N and 5 N floats, and the pointer is made opaque after each step so that the 32 row
  // addresses are not turned into 32 loop-invariant offsets held in registers.
  const bool full = r0 + BR <= R;
  const uint32_t voff = (uint32_t)((4 * lh * N + l32) * 4);
  const int64_t step1 = (int64_t)N * 4, step5 = (int64_t)N * 20;
  auto store_impl = [&](float* out_rows /* row r0 of the output */, const float* res_rows, auto&& value, auto has_res)
      __attribute__((always_inline)) {
    if (!col_ok) return;
    gchar* rowp = (gchar*)(out_rows + (int64_t)wrow * N + wcol);
    const gchar* resp = nullptr;
    if constexpr (decltype(has_res)::value) resp = (const gchar*)(res_rows + (int64_t)wrow * N + wcol);
    if (full) {
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float v = value(t, r);
          if constexpr (decltype(has_res)::value) v += *(const gfloat*)(resp + voff);
          *(gfloat*)(rowp + voff) = v;
          const int64_t st = (r % 4 == 3) ? step5 : step1;
          rowp += st;
          asm volatile("" : "+s"(rowp));
          if constexpr (decltype(has_res)::value) {
            resp += st;
            asm volatile("" : "+s"(resp));
          }
        }
    } else {
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = t * 32 + 8 * (r / 4) + r % 4;
          if (r0 + wrow + row + 4 * lh < R) {
            float v = value(t, r);
            if constexpr (decltype(has_res)::value) v += *(const gfloat*)(resp + voff);
            *(gfloat*)(rowp + voff) = v;
          }
          const int64_t st = (r % 4 == 3) ? step5 : step1;
          rowp += st;
          asm volatile("" : "+s"(rowp));
          if constexpr (decltype(has_res)::value) {
            resp += st;
            asm volatile("" : "+s"(resp));
          }
        }
    }
  };
  // res_rows = row r0 of the matching residual array, or nullptr (the same for the whole workgroup)
  auto store = [&](float* out_rows, const float* res_rows, auto&& value) __attribute__((always_inline)) {
    if (res_rows != nullptr) store_impl(out_rows, res_rows, value, std::true_type{});
    else store_impl(out_rows, res_rows, value, std::false_type{});
  };

  float d1[TM][16], d2[TM][16], ssq[TM][16];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) ssq[t][r] = 0.f;

  // One step: ask for the next tile, multiply the current one, wait for the loads (and for the
  // previous step's stores), and only then store; the barrier also says that every wavefront
  // is done reading the buffer that the step after this one refills.
  auto product = [&](int it, const float* cur, float* nxt, floatx16 (&acc)[TM]) __attribute__((always_inline)) {
    if (it + 1 < n_iter) issue(tile_src(it + 1), nxt);
    compute(cur, acc);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  auto jac_step = [&](int it, const float* cur, float* nxt) __attribute__((always_inline)) {
    floatx16 acc[TM];
    product(it, cur, nxt, acc);
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) ssq[t][r] += acc[t][r] * acc[t][r];
    const int64_t joff = ((int64_t)(p0 + it - 1) * R + r0) * N;
    store(a.y_jac + joff, a.res_jac ? a.res_jac + joff : nullptr, [&](int t, int r) { return d1[t][r] * acc[t][r]; });
  };
  auto lap_step = [&](const float* cur) __attribute__((always_inline)) {
    floatx16 acc[TM];
    compute(cur, acc);
    store(a.y_lap + r0 * N, a.res_lap ? a.res_lap + r0 * N : nullptr,
          [&](int t, int r) { return d1[t][r] * acc[t][r] + d2[t][r] * ssq[t][r]; });
  };

  issue(tile_src(0), As0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  {
    floatx16 acc[TM];
    product(0, As0, As1, acc);
    float o[TM][16];
#define FOLX_DA_CASE(A)                                                                      \
  case A:                                                                                    \
    _Pragma("unroll") for (int t = 0; t < TM; ++t) _Pragma("unroll") for (int r = 0; r < 16; ++r) \
        act_eval<A>(acc[t][r] + bcol, a.prm, o[t][r], d1[t][r], d2[t][r]);                    \
    break;
    switch (a.act) {
      FOLX_DA_CASE(FOLX_ACT_TANH) FOLX_DA_CASE(FOLX_ACT_SILU) FOLX_DA_CASE(FOLX_ACT_LOGISTIC)
      FOLX_DA_CASE(FOLX_ACT_SOFTPLUS) FOLX_DA_CASE(FOLX_ACT_EXP) FOLX_DA_CASE(FOLX_ACT_SIN)
      FOLX_DA_CASE(FOLX_ACT_COS) FOLX_DA_CASE(FOLX_ACT_GELU) FOLX_DA_CASE(FOLX_ACT_GELU_TANH)
      default:
        _Pragma("unroll") for (int t = 0; t < TM; ++t) _Pragma("unroll") for (int r = 0; r < 16; ++r)
            act_eval<FOLX_ACT_SQUARE>(acc[t][r] + bcol, a.prm, o[t][r], d1[t][r], d2[t][r]);
        break;
    }
#undef FOLX_DA_CASE
    if (mode == 0 || (mode == 1 && g == 0))
      store(a.y + r0 * N, a.res ? a.res + r0 * N : nullptr, [&](int t, int r) { return o[t][r]; });
  }
  // Jacobian rows: odd steps read As1, even steps As0
  int it = 1;
  for (; it + 1 <= nJ; it += 2) {
    jac_step(it, As1, As0);
    jac_step(it + 1, As0, As1);
  }
  const bool odd = it <= nJ;
  if (odd) jac_step(it, As1, As0);
  float* part = a.part + (int64_t)rt * G * PART_PER_BLOCK;
  if (mode == 1) {
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[(int64_t)g * PART_PER_BLOCK + (t * 16 + r) * NTHR + tid] = ssq[t][r];
    return;
  }
  if (mode == 2) {
    for (int gg = 0; gg < G; ++gg)
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) ssq[t][r] += part[(int64_t)gg * PART_PER_BLOCK + (t * 16 + r) * NTHR + tid];
  }
  // the lap tile was requested by the last step before it and has been waited for
  if (odd) lap_step(As0); else lap_step(As1);
}

// Few Jacobian rows (P <= 6: networks whose Jacobian stays sparse per node, pair features of FermiNet-style layers).  The
// kernel above walks such a layer in P + 2 dependent steps of one 32-row tile, each behind a barrier, so a small batch took
// that chain's latency on a quarter of the CUs.  Here a workgroup owns 16 to 128 positions and asks for all P + 2 tiles at
// once, waits once, and each wavefront forms its 16 x 16 block of every one of the P + 2 products side by side
// (v_mfma_f32_16x16x4_f32: independent accumulators of 4 registers, one W operand for all of them, taken from L2 16 k
// ahead), which leaves f', f'' and the sum of squares as plain register arithmetic.  The product is formed transposed, so
// a lane holds 4 consecutive columns of one position and stores them 128 bits at a time.  LDS tiles as above, one per row s
// of the triplet; 40 to 88 VGPRs (P = 0 .. 6).  The products of a column are added in the order of the kernel above (128-bit reads of 16 k in
// another order took 1 us less a layer and stood further from 64 bits on a small FermiNet-style function).  A form with W in registers, a grid of the resident workgroups and
// the next tile's loads behind the current product was no faster on large R (28 .. 40 % slower for P = 6) and 15 % slower on
// small.
// us, general kernel -> this: R = 2000, P = 4, 100 x 100: 18.7 -> 11.7; 300, 2, 16 x 16: 8.6 -> 4.0; 25 088, 6, 32 x 32 with a
// skip connection: 50 -> 20 (4 TB/s); 262 144 of these: 260 -> 167 (4.8 TB/s).
template <int NR>
__global__ __launch_bounds__(512) void dense_act_few_kernel(DAParams a, int wc, int wr, int vec) {
  extern __shared__ __attribute__((aligned(16))) float tile[];
  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l16 = lane % 16;
  const int lq = lane / 16;
  const int K = a.K, N = a.N;
  const int npr = K / 4;
  const int64_t R = a.R, RK = R * K;
  const int br = 16 * wr;
  const int64_t r0 = (int64_t)blockIdx.x * br;

  int sh = __builtin_ctz(npr);
  if (sh > 4) sh = 4;
  const int rshift = 4 - sh;
  const int rmask = (1 << sh) - 1;

  const int pieces = br * npr;
  const int stride = pieces * 4;  // floats from one tile to the next
  for (int c = wave * 64; c < pieces; c += 64 * wc * wr) {
    const int q = c + lane;
    if (q < pieces) {  // lane i's 16 bytes land at slot c + i
      int m = q / npr;
      const int piece = (q - m * npr) ^ ((m >> rshift) & rmask);
      if (r0 + m >= R) m = (int)(R - 1 - r0);
      const int off = m * K + 4 * piece;
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        const float* src = (s == 0 ? a.x : (s < NR - 1 ? a.jac + (s - 1) * RK : a.lap)) + r0 * K;
        __builtin_amdgcn_global_load_lds(FOLX_GPTR(src + off), FOLX_LPTR(&tile[s * stride + c * 4]), 16, 0, 0);
      }
    }
  }

  const int col0 = wave % wc * 16;
  const int row = wave / wc * 16 + l16;  // this lane's position in the tile
  const float* wp = a.W + min(col0 + l16, N - 1);
  const int groups = (K + 7) / 8;
  // k of this lane in step e of group j: 8 j + 4 (lane / 16 % 2) + 2 e + lane / 32, so that a column's products are added in the
  // general kernel's order (two of its steps in one)
  const int k0 = 4 * (lq & 1) + (lq >> 1);
  float w[4];
  auto load_w = [&](int j) __attribute__((always_inline)) {  // groups j and j + 1
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 8 * j + k0 + 8 * (i / 2) + 2 * (i % 2);
      w[i] = k < K ? wp[(int64_t)k * N] : 0.f;
    }
  };
  load_w(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  floatx4 acc[NR];
#pragma unroll
  for (int s = 0; s < NR; ++s) acc[s] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int sw = (row >> rshift) & rmask;
  const float* base = tile + row * K;
  auto group = [&](int j, float w0, float w1) __attribute__((always_inline)) {
    // past K a lane meets zeros of W and the last piece of its own row
    const int at = ((min(2 * j + (lq & 1), npr - 1) ^ sw) * 4) + (lq >> 1);
    float v0[NR], v1[NR];
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      v0[s] = base[s * stride + at];
      v1[s] = base[s * stride + at + 2];
    }
#pragma unroll
    for (int s = 0; s < NR; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0, v0[s], acc[s], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < NR; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1, v1[s], acc[s], 0, 0, 0);
  };
  for (int j = 0; j < groups; j += 2) {
    const float wv[4] = {w[0], w[1], w[2], w[3]};
    if (j + 2 < groups) load_w(j + 2);
    group(j, wv[0], wv[1]);
    if (j + 1 < groups) group(j + 1, wv[2], wv[3]);
  }

  // register r of a 16 x 16 block: position lane % 16, column 4 (lane / 16) + r
  const int n0 = col0 + 4 * lq;
  const int cols = min(4, N - n0);
  if (r0 + row >= R || cols <= 0) return;
  float d1[4], d2[4];
  floatx4 ssq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float o;
    act_eval_fused(a.act, acc[0][r] + ((a.bias != nullptr && r < cols) ? a.bias[n0 + r] : 0.f), a.prm, o, d1[r], d2[r]);
    acc[0][r] = o;
#pragma unroll
    for (int s = 1; s < NR - 1; ++s) {
      ssq[r] += acc[s][r] * acc[s][r];
      acc[s][r] *= d1[r];
    }
    acc[NR - 1][r] = d1[r] * acc[NR - 1][r] + d2[r] * ssq[r];
  }
  const int64_t at = (r0 + row) * N + n0, RN = R * N;
  if (a.res != nullptr) {
    floatx4 rv[NR];
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const float* p = (s == 0 ? a.res : (s < NR - 1 ? a.res_jac + (s - 1) * RN : a.res_lap)) + at;
      if (vec) rv[s] = *reinterpret_cast<const floatx4*>(p);
      else
#pragma unroll
        for (int r = 0; r < 4; ++r) rv[s][r] = r < cols ? p[r] : 0.f;
    }
#pragma unroll
    for (int s = 0; s < NR; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[s][r] += rv[s][r];
  }
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    float* p = (s == 0 ? a.y : (s < NR - 1 ? a.y_jac + (s - 1) * RN : a.y_lap)) + at;
    if (vec) *reinterpret_cast<floatx4*>(p) = acc[s];
    else
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < cols) p[r] = acc[s][r];
  }
}

constexpr int FEW_ROWS = 6;
constexpr int FEW_LDS = 40960;  // four workgroups a CU where several row blocks share one

// When the few-rows kernel is the faster one (both timed over 2100 shapes: R = 55 .. 240 000, K = 4 .. 128, N = 1 .. 128, P = 0 .. 6).
// The general kernel reads W into registers once for all rows of a tile and overlaps its loads with its matrix work, which
// is worth 5 to 25 % once its tiles cover the CUs; below that (160 tiles) the few-rows kernel took 0.43 .. 0.95 of its time, up to 192
// 0.74 .. 0.98 unless all of the general kernel's matrix work is for columns and features that exist (its K comes in five sizes, its
// columns in strips of 32, 64 or 128): 128 x 128 1.04, 1.07, 1.14 for P = 1, 4, 6.  In larger launches it wins where enough of that
// work is padding: 48 x 48 0.81 .. 0.91, 96 x 96 0.84 .. 0.92, K = 128 to N = 64 0.62 .. 0.81, but 100 x 100 0.95 .. 1.03 (112 columns for
// 128).  Its six rows with a share above 0.7 did not (N = 48, K = 32: 1.11 .. 1.20; 84 of 128 columns, K = 64: 1.04 .. 1.14), nor did
// K <= 8, where there is little matrix work to save (96 of 128 columns: P = 2 1.02 .. 1.12, P = 6 1.15 .. 1.26; 48 of 64: P = 1, 3
// 0.85 .. 1.04, P = 6 1.06 .. 1.21).  And it reads a skip connection ahead of its stores, 128 bits at a time where N allows: 0.4 .. 1.0
// (once 1.2).  For N not a multiple of 4 its lanes store four single floats, 16 bytes apart from lane to lane: in launches that cover the CUs
// it needs so much more padded work saved per column, the more rows are stored (K, N, P = 20, 42, 5: 1.67; 24, 87, 4: 1.56; 16, 43,
// 1: 1.37; but 124, 41, 6: 0.84; 80, 85, 1: 0.77).
// Of 2100 shapes, skip connections and any N among them, its choice was more than 3 % slower than the general kernel on 28, at most 20 %.
// 300 others without one: 0.69 of the general kernel's time in the mean, 4 to 7 % more on three.
bool few_rows(const DAPlan& pl, int32_t P, int32_t K, int32_t N, bool has_res) {
  if (P > FEW_ROWS) return false;
  if (has_res) return true;
  const int cols = (N + 15) / 16 * 16;
  const double share = (K + 7) / 8 * cols / (32.0 * pl.ks * pl.wc);  // of the general kernel's matrix work that this one does
  if (N % 4 != 0 && N > 16 && pl.row_tiles > 120 && 256 * pl.ks * pl.wc * (1 - share) < (45 + 9 * P) * N) return false;
  if (pl.row_tiles <= 192) return K <= 8 || pl.wc < 4 || pl.row_tiles <= 160 || share <= (P == FEW_ROWS ? 0.9 : 0.95);
  if (12 * cols >= 10 * 32 * pl.wc) return false;
  return share <= 0.7 || (K <= 8 ? pl.wc == 2 && P <= 3 : P < FEW_ROWS);
}

template <int NR>
int launch_few(hipStream_t st, const DAParams& prm) {
  const int wc = (prm.N + 15) / 16;
  auto lds = [&](int wr) { return 64 * wr * prm.K * NR; };  // at most 64 KB for wr = 1
  // 8 wavefronts where N leaves room for several row blocks, but no fewer than two workgroups per CU
  int wr = 8 / wc;
  while (wr > 1 && (lds(wr) > FEW_LDS || (prm.R + 16 * wr - 1) / (16 * wr) < 512)) --wr;
  const int64_t blocks = (prm.R + 16 * wr - 1) / (16 * wr);
  if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
  const int vec = prm.N % 4 == 0 && folx_aligned16(prm.y) && folx_aligned16(prm.y_jac) && folx_aligned16(prm.y_lap) &&
                  folx_aligned16(prm.res) && folx_aligned16(prm.res_jac) && folx_aligned16(prm.res_lap);
  dense_act_few_kernel<NR><<<dim3((unsigned)blocks), dim3(64 * wc * wr), lds(wr), st>>>(prm, wc, wr, vec);
  return folx_launch_status();
}

template <int KS, int WC>
void launch_da(hipStream_t st, DAParams prm, const DAPlan& pl) {
  if (pl.G == 1) {
    prm.mode = 0;
    dense_act_kernel<KS, WC><<<dim3((unsigned)pl.row_tiles), dim3(NTHR), 0, st>>>(prm);
  } else {
    prm.mode = 1;
    dense_act_kernel<KS, WC><<<dim3((unsigned)(pl.row_tiles * pl.G)), dim3(NTHR), 0, st>>>(prm);
    prm.mode = 2;
    dense_act_kernel<KS, WC><<<dim3((unsigned)pl.row_tiles), dim3(NTHR), 0, st>>>(prm);
  }
}

}  // namespace

extern "C" int64_t folx_hip_dense_act_workspace_bytes(int64_t R, int32_t P, int32_t K, int32_t N) {
  DAPlan pl;
  if (R < 0 || P < 0) return FOLX_HIP_EINVAL;
  if (!plan_dense_act(R, P, K, N, pl)) return folx_dense_act_wide_ws_bytes(R, P, K, N);
  return pl.ws_bytes;
}

extern "C" int folx_hip_dense_act_form(int64_t R, int32_t P, int32_t K, int32_t N, int32_t has_res) {
  DAPlan pl;
  if (R <= 0 || P < 0) return FOLX_HIP_EINVAL;
  if (plan_dense_act(R, P, K, N, pl)) return few_rows(pl, P, K, N, has_res != 0) ? FOLX_HIP_FORM_FEW : FOLX_HIP_FORM_TILES;
  return folx_dense_act_wide_group(R, P, K, N);
}

extern "C" int64_t folx_hip_dense_act_pieces_bytes(int64_t R, int32_t P, int32_t K, int32_t N) {
  if (R < 0 || P < 0 || K <= 0 || N <= 0) return FOLX_HIP_EINVAL;
  DAPlan pl;
  return plan_dense_act(R, P, K, N, pl) ? FOLX_HIP_ENOTSUP : folx_wide_pieces_ws_bytes(R, P, K, N);
}

extern "C" int folx_hip_dense_act_pieces_faster(int64_t R, int32_t P, int32_t K, int32_t N, int32_t plain_K) {
  if (R < 0 || P < 0 || K <= 0 || N <= 0 || plain_K <= 0) return FOLX_HIP_EINVAL;
  DAPlan pl;
  return plan_dense_act(R, P, K, N, pl) ? FOLX_HIP_ENOTSUP : folx_wide_pieces_faster(R, P, K, N, plain_K);
}

extern "C" int folx_hip_dense_act_faster(int64_t R, int32_t P, int32_t K, int32_t N, int32_t plain_K) {
  DAPlan pl;
  if (R <= 0 || P < 0 || plain_K <= 0) return FOLX_HIP_EINVAL;
  if (plan_dense_act(R, P, K, N, pl)) return 1;
  return folx_dense_act_wide_faster(R, P, K, N, plain_K);
}

extern "C" int folx_hip_dense_act_fwdlap(void* stream, int32_t act, float param, const float* x, const float* jac,
                                         const float* lap, const float* W, const float* bias, const float* res,
                                         const float* res_jac, const float* res_lap, float* y,
                                         float* y_jac, float* y_lap, int64_t R, int32_t P, int32_t K, int32_t N,
                                         void* workspace, int64_t workspace_bytes) {
  if (R < 0 || P < 0 || K <= 0 || N <= 0) return FOLX_HIP_EINVAL;
  if ((res != nullptr) != (res_lap != nullptr) || (P > 0 && (res != nullptr) != (res_jac != nullptr)))
    return FOLX_HIP_EINVAL;
  if (!act_fused(act)) return FOLX_HIP_ENOTSUP;
  DAPlan pl;
  if (!plan_dense_act(R, P, K, N, pl)) {
    if (res) return FOLX_HIP_ENOTSUP;  // the wide path adds a skip connection only when it reads its operand in parts
    return folx_dense_act_wide((hipStream_t)stream, act, param, x, jac, lap, W, bias, y, y_jac, y_lap, R, P, K, N,
                               workspace, workspace_bytes);
  }
  if (R == 0) return FOLX_HIP_OK;
  if (!x || !lap || !W || !y || !y_lap || (P > 0 && (!jac || !y_jac))) return FOLX_HIP_EINVAL;
  if (!folx_aligned16(x) || !folx_aligned16(lap) || (P > 0 && !folx_aligned16(jac))) return FOLX_HIP_ENOTSUP;
  if (pl.ws_bytes > 0 && (!workspace || workspace_bytes < pl.ws_bytes || !folx_aligned16(workspace)))
    return FOLX_HIP_EINVAL;
  DAParams prm;
  prm.x = x; prm.jac = jac; prm.lap = lap; prm.W = W; prm.bias = bias;
  prm.res = res; prm.res_jac = res_jac; prm.res_lap = res_lap;
  prm.y = y; prm.y_jac = y_jac; prm.y_lap = y_lap;
  prm.part = (float*)workspace;
  prm.R = R; prm.P = P; prm.K = K; prm.N = N; prm.G = pl.G; prm.PG = pl.PG; prm.act = act; prm.prm = param; prm.mode = 0;
  hipStream_t st = (hipStream_t)stream;
  switch (few_rows(pl, P, K, N, res != nullptr) ? P : FEW_ROWS + 1) {
    case 0: return launch_few<2>(st, prm);
    case 1: return launch_few<3>(st, prm);
    case 2: return launch_few<4>(st, prm);
    case 3: return launch_few<5>(st, prm);
    case 4: return launch_few<6>(st, prm);
    case 5: return launch_few<7>(st, prm);
    case FEW_ROWS: return launch_few<8>(st, prm);
    default: break;
  }
  const int code = pl.wc * 100 + pl.ks;
  switch (code) {
    case 101: launch_da<1, 1>(st, prm, pl); break;
    case 104: launch_da<4, 1>(st, prm, pl); break;
    case 201: launch_da<1, 2>(st, prm, pl); break;
    case 204: launch_da<4, 2>(st, prm, pl); break;
    case 208: launch_da<8, 2>(st, prm, pl); break;
    case 401: launch_da<1, 4>(st, prm, pl); break;
    case 404: launch_da<4, 4>(st, prm, pl); break;
    case 408: launch_da<8, 4>(st, prm, pl); break;
    case 413: launch_da<13, 4>(st, prm, pl); break;
    case 416: launch_da<16, 4>(st, prm, pl); break;
    default: return FOLX_HIP_ENOTSUP;
  }
  return folx_launch_status();
}
