// Matrix product of two operands that BOTH carry derivatives (attention scores q k^T, p v
// written with plain matmul / einsum):
//
//   y        = a b
//   y_jac[p] = a_jac[p] b + a b_jac[p]
//   y_lap    = a_lap b + a b_lap + 2 sum_p a_jac[p] b_jac[p]
//
// for a batch of small matrices, a (I x Kc), b (Kc x J), every operand addressed through element
// strides so that transposed and head-interleaved views ((walker, electron, head, feature)
// read as (walker, head, electron, feature)) are consumed where they lie.  The
// (batch, i, j, k) intermediate of the multiply-and-sum decomposition is never formed: per
// Jacobian row the kernel reads one (I x Kc) and one (Kc x J) tile and writes one (I x J) tile.
//
// One workgroup of four wavefronts per (batch element, 32 x 32 output tile); wavefront w owns
// the 16 x 16 block (w / 2, w % 2).  a and b tiles stay in LDS for the whole Jacobian loop, the
// row's a_jac[p] / b_jac[p] tiles are fetched into registers one row ahead and handed over
// through LDS; three v_mfma_f32_16x16x4_f32 chains per row (a_jac b, a b_jac into the row's
// accumulator, a_jac b_jac into the Laplacian's).  The Laplacian operands run through the same
// loop body as one more row (p = P) that is left out of the second-order sum.  Inside a group of
// 16 values of k the order is permuted (lane (l16, lg), step r <-> k = 4 lg + r), so the A
// operand is one 128-bit LDS read per four MFMAs.
//
// Up to 32 x 32 x 32 nothing has to be shared: dot_two_small_kernel (its mapping stands there).

#include "common.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int DT_TILE = 32;    // output tile edge
constexpr int DT_NT = 256;     // threads per workgroup
constexpr int DT_KMAX = 128;   // contracted length the LDS tiles are sized for
constexpr int DT_BS = 48;      // row stride of the (k x 32) tiles: 16 mod 32, two k rows per half wavefront hit disjoint banks

struct DotTwoArgs {
  const float *a, *aj, *al, *b, *bj, *bl;
  float *y, *yj, *yl;
  // element strides: batch index = b0 * NB1 + b1
  int64_t a_sb0, a_sb1, a_si, a_sk, a_sp;
  int64_t b_sb0, b_sb1, b_sk, b_sj, b_sp;
  int64_t y_sp;  // elements between consecutive Jacobian rows of y_jac (= NB * I * J)
  int64_t NB;
  int32_t NB1, I, J, Kc, P, tiles_i, tiles_j;
};

// MAXLD = values per thread of one tile: 32 * Kp / 256 with Kp = Kc rounded up to 16
// CONSTB: b carries no derivatives (a constant with batch axes, e.g. per-head weights): the rule is
// linear in a, y_jac[p] = a_jac[p] b and y_lap = a_lap b, one product chain per row and no b rows.
template <int MAXLD, bool CONSTB>
__global__ __launch_bounds__(DT_NT) void dot_two_kernel(DotTwoArgs g) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int Kc = g.Kc;
  const int Kp = (Kc + 15) / 16 * 16;
  const int AS = Kp + 4;                      // row stride of the (32 x k) tiles
  float* As = sm;                             // a        [32][AS]
  float* AJs = As + DT_TILE * AS;             // a_jac[p] [32][AS]
  float* Bs = AJs + DT_TILE * AS;             // b        [Kp][DT_BS]
  float* BJs = Bs + Kp * DT_BS;               // b_jac[p] [Kp][DT_BS]

  const int tid = threadIdx.x;
  const int lane = tid % FOLX_WAVE, w = tid / FOLX_WAVE;
  const int l16 = lane % 16, lg = lane / 16;
  const int wi = w / 2, wj = w % 2;

  int64_t blk = blockIdx.x;
  const int tj = (int)(blk % g.tiles_j); blk /= g.tiles_j;
  const int ti = (int)(blk % g.tiles_i); blk /= g.tiles_i;
  const int64_t bt = blk;
  const int64_t b0 = bt / g.NB1, b1 = bt % g.NB1;
  const int i0 = ti * DT_TILE, j0 = tj * DT_TILE;
  const int64_t a_off = b0 * g.a_sb0 + b1 * g.a_sb1;
  const int64_t b_off = b0 * g.b_sb0 + b1 * g.b_sb1;
  const int nld = DT_TILE * Kp / DT_NT;       // values per thread and tile (Kp / 8)
  // the unit-stride axis of an operand is walked by consecutive threads
  const bool a_kfast = g.a_sk == 1 || g.a_si != 1;
  const bool b_jfast = g.b_sj == 1 || g.b_sk != 1;

  // element e of thread's r-th value -> (row, k) of the a-type tile, (k, col) of the b-type tile
  auto a_coord = [&](int r, int& i, int& k) {
    const int e = tid + DT_NT * r;
    if (a_kfast) { k = e % Kp; i = e / Kp; } else { i = e % DT_TILE; k = e / DT_TILE; }
  };
  auto b_coord = [&](int r, int& k, int& j) {
    const int e = tid + DT_NT * r;
    if (b_jfast) { j = e % DT_TILE; k = e / DT_TILE; } else { k = e % Kp; j = e / Kp; }
  };
  auto fetch_a = [&](const float* src, float (&reg)[MAXLD]) {
#pragma unroll
    for (int r = 0; r < MAXLD; ++r) {
      reg[r] = 0.0f;
      if (r < nld) {
        int i, k;
        a_coord(r, i, k);
        if (i0 + i < g.I && k < Kc) reg[r] = src[a_off + (int64_t)(i0 + i) * g.a_si + (int64_t)k * g.a_sk];
      }
    }
  };
  auto fetch_b = [&](const float* src, float (&reg)[MAXLD]) {
#pragma unroll
    for (int r = 0; r < MAXLD; ++r) {
      reg[r] = 0.0f;
      if (r < nld) {
        int k, j;
        b_coord(r, k, j);
        if (j0 + j < g.J && k < Kc) reg[r] = src[b_off + (int64_t)k * g.b_sk + (int64_t)(j0 + j) * g.b_sj];
      }
    }
  };
  auto put_a = [&](float* dst, const float (&reg)[MAXLD]) {
#pragma unroll
    for (int r = 0; r < MAXLD; ++r)
      if (r < nld) { int i, k; a_coord(r, i, k); dst[i * AS + k] = reg[r]; }
  };
  auto put_b = [&](float* dst, const float (&reg)[MAXLD]) {
#pragma unroll
    for (int r = 0; r < MAXLD; ++r)
      if (r < nld) { int k, j; b_coord(r, k, j); dst[k * DT_BS + j] = reg[r]; }
  };

  float ra[MAXLD], rb[MAXLD];
  fetch_a(g.a, ra);
  fetch_b(g.b, rb);
  put_a(As, ra);
  put_b(Bs, rb);
  // first row in flight: Jacobian row 0, or the Laplacian operands when there are no rows
  fetch_a(g.P > 0 ? g.aj : g.al, ra);
  if constexpr (!CONSTB) fetch_b(g.P > 0 ? g.bj : g.bl, rb);
  __syncthreads();

  // A operand of step (t, r): tile[16 wi + l16][16 t + 4 lg + r]; B operand: tile[16 t + 4 lg + r][16 wj + l16]
  const float* a_row = As + (16 * wi + l16) * AS + 4 * lg;
  const float* aj_row = AJs + (16 * wi + l16) * AS + 4 * lg;
  const float* b_col = Bs + (4 * lg) * DT_BS + 16 * wj + l16;
  const float* bj_col = BJs + (4 * lg) * DT_BS + 16 * wj + l16;
  const int kt = Kp / 16;

  const int orow = i0 + 16 * wi + 4 * lg, ocol = j0 + 16 * wj + l16;
  auto store_tile = [&](float* dst, const floatx4& c) {
    if (ocol < g.J) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (orow + r < g.I) dst[(bt * g.I + orow + r) * (int64_t)g.J + ocol] = c[r];
    }
  };

  {  // y = a b
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < kt; ++t) {
      const float4 av = *reinterpret_cast<const float4*>(a_row + 16 * t);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, b_col[(16 * t + 0) * DT_BS], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, b_col[(16 * t + 1) * DT_BS], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, b_col[(16 * t + 2) * DT_BS], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, b_col[(16 * t + 3) * DT_BS], acc, 0, 0, 0);
    }
    store_tile(g.y, acc);
  }

  floatx4 lap2 = {0.f, 0.f, 0.f, 0.f};  // sum_p a_jac[p] b_jac[p]
  for (int p = 0; p <= g.P; ++p) {
    put_a(AJs, ra);
    if constexpr (!CONSTB) put_b(BJs, rb);
    __syncthreads();
    if (p < g.P) {  // next row: Jacobian row p + 1, or the Laplacian operands after the last one
      const bool last = p + 1 == g.P;
      fetch_a(last ? g.al : g.aj + (int64_t)(p + 1) * g.a_sp, ra);
      if constexpr (!CONSTB) fetch_b(last ? g.bl : g.bj + (int64_t)(p + 1) * g.b_sp, rb);
    }
    floatx4 acc = {0.f, 0.f, 0.f, 0.f}, cross = {0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < kt; ++t) {
      const float4 av = *reinterpret_cast<const float4*>(a_row + 16 * t);
      const float4 ajv = *reinterpret_cast<const float4*>(aj_row + 16 * t);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float bv = b_col[(16 * t + r) * DT_BS];
        const float ajr = r == 0 ? ajv.x : (r == 1 ? ajv.y : (r == 2 ? ajv.z : ajv.w));
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ajr, bv, acc, 0, 0, 0);
        if constexpr (!CONSTB) {
          const float bjv = bj_col[(16 * t + r) * DT_BS];
          const float ar = r == 0 ? av.x : (r == 1 ? av.y : (r == 2 ? av.z : av.w));
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ar, bjv, acc, 0, 0, 0);
          cross = __builtin_amdgcn_mfma_f32_16x16x4f32(ajr, bjv, cross, 0, 0, 0);
        }
      }
    }
    if (p < g.P) {
      lap2 += cross;
      store_tile(g.yj + (int64_t)p * g.y_sp, acc);
    } else {
      store_tile(g.yl, acc + 2.0f * lap2);
    }
    __syncthreads();  // everyone is done with this row's tiles
  }
}

// I, J, Kc <= 32: one wavefront covers a whole batch element (TI x TJ blocks of 16 x 16, KT groups of 16 k), so nothing is
// shared: operands go from memory straight into MFMA operand registers and the W wavefronts of a workgroup take the Jacobian
// rows p = w, w + W, ..., the next row's operands requested before this row's products; the sums over rows meet in LDS once
// at the end.  The product is formed transposed (b in the A operand), so a lane ends with four consecutive columns of a row
// of y: 128-bit stores.  Padding is lanes whose buffer offset lies past the descriptor's end (zeros; dropped stores).
// a_vec / b_vec: the contracted axis has unit stride and every piece of four is whole and aligned: 128-bit loads.
// Bound by HBM (5.2 TB/s for 16 384 of 16 x 16 x 16, P = 48, 5.1 for 4096 of 32 x 32 x 32, P = 96), for few batch elements by the
// latency of a wavefront's rows.  The tiled form above left three of its four wavefronts without a block and paid two
// barriers and an LDS round trip per row at these sizes: 2048 products of 16 x 16 x 16, P = 48: 336 -> 55 us for b = k^T, 355 -> 55 for
// b row by row; of 32 x 32 x 32, P = 96: 1445 -> 491; 64 of 16 x 16 x 16, P = 48: 102 -> 8; with a constant b 78 -> 34, 387 -> 346, 35 -> 6.
// 300 random sizes up to the limit: 0.08 .. 0.85 of the tiled form's time.
constexpr int NXCD = 8;
constexpr uint32_t FAR = 0x40000000u;      // past every descriptor's end
constexpr int64_t EXTENT_MAX = 0x0fffffff;  // elements of an operand's tile from its first to its last: below FAR in bytes
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

template <int TI, int TJ, int KT, bool CONSTB>
__global__ __launch_bounds__(512) void dot_two_small_kernel(DotTwoArgs g, int a_vec, int b_vec, int y_vec) {
  extern __shared__ __attribute__((aligned(16))) float sm[];  // [W - 1][TI * TJ * 4][64] sums
  const int W = blockDim.x / FOLX_WAVE;
  const int lane = threadIdx.x % FOLX_WAVE, w = folx_wave_id();
  const int l16 = lane % 16, lg = lane / 16;
  // ids are dealt round-robin to the XCDs: consecutive batch elements (heads of a walker share cache lines) go to one
  const int64_t per = (g.NB + NXCD - 1) / NXCD;
  const int64_t bt = (int64_t)(blockIdx.x % NXCD) * per + blockIdx.x / NXCD;
  if (bt >= g.NB) return;
  const int64_t b0 = bt / g.NB1, b1 = bt % g.NB1;
  const int I = g.I, J = g.J, Kc = g.Kc, P = g.P;
  const int64_t a_off = b0 * g.a_sb0 + b1 * g.a_sb1, b_off = b0 * g.b_sb0 + b1 * g.b_sb1;
  const uint32_t a_si = (uint32_t)g.a_si, a_sk = (uint32_t)g.a_sk, b_sj = (uint32_t)g.b_sj, b_sk = (uint32_t)g.b_sk;
  const uint32_t a_bytes = Kc > 0 ? 4u * ((uint32_t)(I - 1) * a_si + (uint32_t)(Kc - 1) * a_sk + 1u) : 0u;
  const uint32_t b_bytes = Kc > 0 ? 4u * ((uint32_t)(J - 1) * b_sj + (uint32_t)(Kc - 1) * b_sk + 1u) : 0u;

  // element (row / column l16 of block i, k = 16 t + 4 lg + r)
  auto load = [&](const float* src, uint32_t bytes, int n, uint32_t s, uint32_t sk, int vec, int blk,
                  floatx4 (&reg)[KT]) __attribute__((always_inline)) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, bytes, 0x00027000);
    const int row = 16 * blk + l16;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int k = 16 * t + 4 * lg;
      const uint32_t base = 4u * ((uint32_t)row * s + (uint32_t)k * sk);
      if (vec) {
        reg[t] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, row < n && k < Kc ? base : FAR, 0, 0));
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          reg[t][r] = __uint_as_float(
              __builtin_amdgcn_raw_buffer_load_b32(rs, row < n && k + r < Kc ? base + 4u * r * sk : FAR, 0, 0));
      }
    }
  };
  auto load_a = [&](const float* src, floatx4 (&reg)[TI][KT]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i) load(src + a_off, a_bytes, I, a_si, a_sk, a_vec, i, reg[i]);
  };
  auto load_b = [&](const float* src, floatx4 (&reg)[TJ][KT]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < TJ; ++j) load(src + b_off, b_bytes, J, b_sj, b_sk, b_vec, j, reg[j]);
  };
  auto store = [&](float* dst, const floatx4 (&c)[TI][TJ]) __attribute__((always_inline)) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(dst + bt * I * J, 0, (uint32_t)(I * J) * 4u, 0x00027000);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int row = 16 * i + l16, col = 16 * j + 4 * lg;
        const uint32_t off = (uint32_t)(row * J + col) * 4u;
        if (y_vec) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, c[i][j]), rs, row < I && col < J ? off : FAR, 0, 0);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = c[i][j][r];
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, row < I && col + r < J ? off + 4u * r : FAR, 0, 0);
          }
        }
      }
  };
  auto mul = [&](const floatx4 (&x)[TI][KT], const floatx4 (&y)[TJ][KT], floatx4 (&acc)[TI][TJ]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[j][t][r], x[i][t][r], acc[i][j], 0, 0, 0);
  };
  auto zero = [&](floatx4 (&acc)[TI][TJ]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  };

  // pass p < P: Jacobian row p; pass p == P: the Laplacians take the place of the row
  floatx4 an[TI][KT], bn[TJ][KT];
  auto fetch = [&](int p) __attribute__((always_inline)) {
    load_a(p == P ? g.al : g.aj + (int64_t)p * g.a_sp, an);
    if constexpr (!CONSTB) load_b(p == P ? g.bl : g.bj + (int64_t)p * g.b_sp, bn);
  };
  floatx4 a[TI][KT], b[TJ][KT], cross[TI][TJ], lap[TI][TJ];
  load_a(g.a, a);
  load_b(g.b, b);
  if (w <= P) fetch(w);
  if (w == 0) {
    floatx4 acc[TI][TJ];
    zero(acc);
    mul(a, b, acc);
    store(g.y, acc);
  }
  zero(cross);
  zero(lap);
  for (int p = w; p <= P; p += W) {
    floatx4 aj[TI][KT], bj[TJ][KT], acc[TI][TJ];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
#pragma unroll
      for (int i = 0; i < TI; ++i) aj[i][t] = an[i][t];
      if constexpr (!CONSTB)
#pragma unroll
        for (int j = 0; j < TJ; ++j) bj[j][t] = bn[j][t];
    }
    if (p + W <= P) fetch(p + W);
    zero(acc);
    mul(aj, b, acc);
    if constexpr (!CONSTB) {
      mul(a, bj, acc);
      if (p < P) mul(aj, bj, cross);
    }
    if (p < P) {
      store(g.yj + (int64_t)p * g.y_sp, acc);
    } else {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) lap[i][j] = acc[i][j];
    }
  }

  // sums over rows: wavefronts 1 .. W - 1 leave theirs in LDS, wavefront 0 adds them in order
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) lap[i][j][r] += 2.0f * cross[i][j][r];
  if (w > 0) {
    float* o = sm + (w - 1) * (TI * TJ * 4 * FOLX_WAVE) + lane;
#pragma unroll
    for (int e = 0; e < TI * TJ * 4; ++e) o[e * FOLX_WAVE] = lap[e / 4 / TJ][e / 4 % TJ][e % 4];
  }
  __syncthreads();
  if (w > 0) return;
  for (int v = 0; v < W - 1; ++v) {
    const float* o = sm + v * (TI * TJ * 4 * FOLX_WAVE) + lane;
#pragma unroll
    for (int e = 0; e < TI * TJ * 4; ++e) lap[e / 4 / TJ][e / 4 % TJ][e % 4] += o[e * FOLX_WAVE];
  }
  store(g.yl, lap);
}

template <int TI, int TJ, int KT>
int launch_small(hipStream_t st, const DotTwoArgs& g, bool constb, int a_vec, int b_vec, int y_vec) {
  // Fewer than eight rows are not worth sharing in launches that fill the chip; eight wavefronts where a CU gets one batch element
  // at most.  us for W = 1, 4, 8, 16 x 16 x 16: 192, P = 16: 11.0, 6.3, 6.0; P = 48: 25.2, 10.3, 9.0; 512, P = 48: 26.9, 14.1, 13.1.  32 x 32 x 32:
  // 192, P = 16: 37.5, 16.9, 17.0; P = 48: 98, 34.5, 32.4; 512, P = 48: 102, 55.2, 59.5; few elements with few rows would be
  // faster with four (64, P = 6: 17.8, 9.6).
  const int W = g.P < 8 ? 1 : (g.NB <= 192 && g.P >= 16 ? 8 : 4);
  const size_t lds = sizeof(float) * (W - 1) * TI * TJ * 4 * FOLX_WAVE;
  const dim3 grid((unsigned)((g.NB + NXCD - 1) / NXCD * NXCD)), block((unsigned)(FOLX_WAVE * W));
  if (constb) dot_two_small_kernel<TI, TJ, KT, true><<<grid, block, lds, st>>>(g, a_vec, b_vec, y_vec);
  else dot_two_small_kernel<TI, TJ, KT, false><<<grid, block, lds, st>>>(g, a_vec, b_vec, y_vec);
  return folx_launch_status();
}

}  // namespace

extern "C" int folx_hip_dot_two_fwdlap(void* stream, const float* a, const float* a_jac, const float* a_lap,
                                       const float* b, const float* b_jac, const float* b_lap, float* y,
                                       float* y_jac, float* y_lap, int64_t NB0, int32_t NB1, int32_t I,
                                       int32_t J, int32_t Kc, int32_t P, const int64_t* strides) {
  if (NB0 < 0 || NB1 < 0 || I < 0 || J < 0 || Kc < 0 || P < 0 || !strides) return FOLX_HIP_EINVAL;
  if (Kc > DT_KMAX) return FOLX_HIP_ENOTSUP;
  const int64_t NB = NB0 * NB1;
  if (NB == 0 || I == 0 || J == 0) return FOLX_HIP_OK;
  const bool constb = !b_jac && !b_lap;  // b without derivatives
  if (!a || !a_lap || !b || !y || !y_lap || (P > 0 && (!a_jac || !y_jac))) return FOLX_HIP_EINVAL;
  if (!constb && (!b_lap || (P > 0 && !b_jac))) return FOLX_HIP_EINVAL;
  DotTwoArgs g;
  g.a = a; g.aj = a_jac; g.al = a_lap; g.b = b; g.bj = b_jac; g.bl = b_lap;
  g.y = y; g.yj = y_jac; g.yl = y_lap;
  g.a_sb0 = strides[0]; g.a_sb1 = strides[1]; g.a_si = strides[2]; g.a_sk = strides[3]; g.a_sp = strides[4];
  g.b_sb0 = strides[5]; g.b_sb1 = strides[6]; g.b_sk = strides[7]; g.b_sj = strides[8]; g.b_sp = strides[9];
  for (int i = 0; i < 10; ++i)
    if (strides[i] < 0) return FOLX_HIP_EINVAL;
  g.NB = NB; g.NB1 = NB1; g.I = I; g.J = J; g.Kc = Kc; g.P = P;
  g.y_sp = NB * (int64_t)I * J;
  hipStream_t st = (hipStream_t)stream;
  const int64_t a_ext = (I - 1) * g.a_si + (Kc > 0 ? Kc - 1 : 0) * g.a_sk, b_ext = (J - 1) * g.b_sj + (Kc > 0 ? Kc - 1 : 0) * g.b_sk;
  if (I <= 32 && J <= 32 && Kc <= 32 && a_ext < EXTENT_MAX && b_ext < EXTENT_MAX && NB <= 0x7ffffff0LL) {
    const bool whole = Kc % 4 == 0;
    const int a_vec = whole && g.a_sk == 1 && ((g.a_si | g.a_sb0 | g.a_sb1 | g.a_sp) & 3) == 0 && folx_aligned16(a) &&
                      folx_aligned16(a_jac) && folx_aligned16(a_lap);
    const int b_vec = whole && g.b_sk == 1 && ((g.b_sj | g.b_sb0 | g.b_sb1 | g.b_sp) & 3) == 0 && folx_aligned16(b) &&
                      folx_aligned16(b_jac) && folx_aligned16(b_lap);
    const int y_vec = J % 4 == 0 && folx_aligned16(y) && folx_aligned16(y_jac) && folx_aligned16(y_lap);
    const int form = (I > 16 ? 4 : 0) + (J > 16 ? 2 : 0) + (Kc > 16 ? 1 : 0);
    switch (form) {
      case 0: return launch_small<1, 1, 1>(st, g, constb, a_vec, b_vec, y_vec);
      case 1: return launch_small<1, 1, 2>(st, g, constb, a_vec, b_vec, y_vec);
      case 2: return launch_small<1, 2, 1>(st, g, constb, a_vec, b_vec, y_vec);
      case 3: return launch_small<1, 2, 2>(st, g, constb, a_vec, b_vec, y_vec);
      case 4: return launch_small<2, 1, 1>(st, g, constb, a_vec, b_vec, y_vec);
      case 5: return launch_small<2, 1, 2>(st, g, constb, a_vec, b_vec, y_vec);
      case 6: return launch_small<2, 2, 1>(st, g, constb, a_vec, b_vec, y_vec);
      default: return launch_small<2, 2, 2>(st, g, constb, a_vec, b_vec, y_vec);
    }
  }
  g.tiles_i = (I + DT_TILE - 1) / DT_TILE;
  g.tiles_j = (J + DT_TILE - 1) / DT_TILE;
  const int64_t blocks = NB * g.tiles_i * g.tiles_j;
  if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
  const int Kp = (Kc + 15) / 16 * 16 > 0 ? (Kc + 15) / 16 * 16 : 16;
  g.Kc = Kc;
  const size_t lds = sizeof(float) * (2 * DT_TILE * (Kp + 4) + 2 * Kp * DT_BS);
  const int nld = DT_TILE * Kp / DT_NT;  // 2, 4, ..., 16
  const dim3 grid((unsigned)blocks), block(DT_NT);
  if (nld <= 4) {
    if (constb) dot_two_kernel<4, true><<<grid, block, lds, st>>>(g);
    else dot_two_kernel<4, false><<<grid, block, lds, st>>>(g);
  } else if (nld <= 8) {
    if (constb) dot_two_kernel<8, true><<<grid, block, lds, st>>>(g);
    else dot_two_kernel<8, false><<<grid, block, lds, st>>>(g);
  } else {
    if (lds > 64 * 1024) {
      static FolxLdsGrant grant[2];
      const void* kernel = constb ? reinterpret_cast<const void*>(dot_two_kernel<16, true>)
                                  : reinterpret_cast<const void*>(dot_two_kernel<16, false>);
      if (!grant[constb ? 1 : 0].ask(kernel, 96 * 1024)) return FOLX_HIP_ENOTSUP;
    }
    if (constb) dot_two_kernel<16, true><<<grid, block, lds, st>>>(g);
    else dot_two_kernel<16, false><<<grid, block, lds, st>>>(g);
  }
  return folx_launch_status();
}
