// Wide dense layer (N > 128, K a multiple of 16) with the elementwise work around it folded
// into the GEMM over the Jacobian rows, so that neither the pre-activation Jacobian nor a
// normalised copy of the input Jacobian goes through HBM:
//
//   (a) dense + activation                    y = f(x @ W + bias)
//   (b) LayerNorm + dense                     y = LN(x) @ W + bias
//   (c) LayerNorm + dense + activation        y = f(LN(x) @ W + bias)
//
// with LN(x) = gamma * xh + beta, xh = (x - mean) * rs, rs = rsqrt(var + eps) over the K
// features of a position.  The Jacobian rows are (P * R) x K with R positions.
//
// Activation.  With z = ... @ W + bias, zj[p] and zl the pre-activation triplet,
//   y = f(z),  yj[p] = f'(z) zj[p],  yl = f'(z) zl + f''(z) sum_p zj[p]^2.
//
// LayerNorm in front of a matrix product.  For a Jacobian row t (K features of one position)
// with a = mean(t), b = mean(xh t):   LN'[t] = gamma rs (t - a - b xh), hence
//   LN'[t] @ W = rs (t @ Wg - a w1 - b w2),   Wg = diag(gamma) W,  w1 = 1^T Wg,  w2 = xh @ Wg,
// a rank-2 correction of the product of the RAW row with Wg; w2 = z - bias - beta @ W is known
// from the x row.  The second-order term of LayerNorm, summed over Jacobian rows,
//   rs^2 gamma (-2 V + xh (3 sum_p b_p^2 - sum_p q_p)),  V = sum_p b_p (t_p - a_p),
//   q_p = mean(t_p^2) - a_p^2,
// goes through W as  rs^2 (-2 sum_p b_p (t_p @ Wg - a_p w1) + w2 (3 sum b^2 - sum q)).
// a_p, b_p and mean(t_p^2) are summed from the A tile while it feeds the MFMAs.
//
// Launches on the caller's stream:
//  1. (LayerNorm only) fold gamma / beta into the weights (the pieces of Wg, w1, c0 = bias + beta @ W), and
//     one wavefront per position for xh, rs and the linear part of LN's lap row before gamma;
//  2. the plain dense kernel on the x and lap rows only (2 R of the (P + 2) R rows; xh @ Wg + c0 behind LayerNorm): z goes to
//     y, the linear part of zl to y_lap; without LayerNorm it leaves the pieces of W as well;
//  3. the Jacobian GEMM below, whose 128-row tiles are cut ACROSS Jacobian rows: a tile holds
//     4 consecutive positions x 32 consecutive p, ordered position-major, so that each 32 x 32
//     accumulator block belongs to ONE position.  f'(z), w1, w2 and rs of a block are then one
//     value per lane (its column), and the sums over p inside a block stay inside the
//     wavefront (16 registers and the two lane halves).  The sums go to the workspace, one
//     (R, N) slab per group of 32 Jacobian rows;
//  4. a short elementwise kernel that finishes y and y_lap, adding the slabs in a fixed order.
//
// Variant (a) also reads a CONCATENATED operand part by part (a chunk of 16 features lies in
// exactly one part; a part may hold one row per walker that all of the walker's positions
// share) and adds a skip connection in its epilogue, so that a layer fed by
// [own features, per-walker means, ...] forms neither the broadcasts nor the concatenation.
//
// The products are SplitTile's (split_bf16.h), a wavefront's 32 rows one position (32 Jacobian rows), two or four; what the epilogue
// needs per position and column (z - c0, f'(z)) waits in LDS.
//
// What bounds it: the power cap, as for the plain product; beyond that, us for K = N = 256, P = 96, 32 768 positions: 2700 behind LayerNorm and
// 2780 with tanh as well against 2330 plain (the row sums and the rank-2 correction are as many vector instructions as the split of A;
// with the fp32 instructions 3670 and 3760).  Read in parts, K = 320, P = 48 in groups of 16, 16 384 positions: 1300 -> 990.
// What the accumulators start from (the per-walker term) has to be put together block by block, and the loop to exist once: the registers
// of two would be spilled (29 -> 25 ms for the whole of such a model).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "activations.h"
#include "dense_act_wide.h"
#include "dense_tiles.h"
#include "split_bf16.h"

namespace {

using folx_split::floatx16;
using folx_split::SplitTile;

constexpr int BK = 16;
constexpr int BM = 128;
constexpr int NXCD = 8;
constexpr int KMAX_NORM = 512; // xh of a tile's positions sits in LDS

using WideParts = FolxWideParts;

struct WideParams {
  const float* jac;
  const char* pieces;  // of W, of Wg with LayerNorm
  const float* z;    // pre-activation values (R, N), bias included
  const float* xhat; // (R, K)           LayerNorm only
  const float* rs;   // (R)
  const float *w1, *c0;  // (N)
  float* y_jac;
  const float* res_jac;  // optional (P, R, N) added to the activated Jacobian rows     PARTS instances only
  const float* pre_jac;  // optional (P, R / pre_group, N) added to the PRE-activation Jacobian rows: position r takes
  int64_t pre_group;     // row r / pre_group (a per-walker term shared by the walker's positions)   PARTS instances only
  float* ss;         // (PG, R, N) sums of zj^2 per group of PT Jacobian rows     activation only
  float* s1;         // (PG, R, N) sums of b_p (t_p @ Wg - a_p w1)                LayerNorm only
  float* sc;         // (PG, R, 2) sums of b_p^2 and of q_p
  int64_t R, row_tiles, pos_tiles;
  int32_t P, K, N, col_tiles, act;
  float prm;
  WideParts parts;   // PARTS instances only (jac unused then)
};

// PT = Jacobian rows of a tile: 32 (4 positions per tile, one per accumulator block), or 16 for
// the activation alone (8 positions per tile, two per block: registers 0-7 of a block belong
// to the first, 8-15 to the second), or 8 (four per block): fewer empty rows (P = 21 fills 24 instead of 32, P = 39 fills 40
// instead of 48 or 64) for more epilogue work per row (act_group).  The activation's tiles may
// hold more positions than are left: those past R read position R - 1 and are neither stored nor summed.
template <int CB, bool NORM, bool ACT, int PT, bool PARTS, bool APART>
__global__ __launch_bounds__(256, 2) void wide_pieces_kernel(WideParams a) {
  static_assert(!PARTS || !NORM, "LayerNorm reads one array");
  using Tile = SplitTile<CB, PARTS, APART>;
  constexpr int BN = Tile::BN;
  constexpr int RT = BM / PT;  // positions of a tile
  constexpr int PB = 32 / PT;  // positions of a wavefront's 32 rows
  static_assert(PT == 32 || ((PT == 16 || PT == 8) && !NORM), "LayerNorm's row sums assume one position per wavefront");
  __shared__ __attribute__((aligned(16))) char ws0[Tile::STAGE];
  __shared__ __attribute__((aligned(16))) char ws1[Tile::STAGE];
  __shared__ __attribute__((aligned(16))) float xhS[NORM ? RT * KMAX_NORM : 4];
  __shared__ __attribute__((aligned(16))) float2 st[NORM ? BM : 1];  // means of a row: (t, xh t)
  __shared__ float w2S[NORM ? RT * BN : 1];  // z - c0 and f'(z) of the tile's positions and columns
  __shared__ float d1S[ACT ? RT * BN : 1];
  __shared__ float w1S[NORM ? BN : 1];

  // ids are dealt round-robin to the XCDs: the column tiles of a row tile stay on one of them
  const int64_t id = blockIdx.x;
  const int64_t xcd = id % NXCD;
  const int64_t slot = id / NXCD;
  const int64_t rt = (slot / a.col_tiles) * NXCD + xcd;
  const int32_t ct = (int32_t)(slot % a.col_tiles);
  if (rt >= a.row_tiles) return;
  const int32_t pg = (int32_t)(rt / a.pos_tiles);
  const int64_t r0 = (rt % a.pos_tiles) * RT;
  const int32_t p0 = pg * PT;
  const int32_t col0 = ct * BN;
  const int32_t K = a.K, N = a.N, P = a.P;
  const int64_t R = a.R;
  auto inside = [&](int64_t pos) __attribute__((always_inline)) -> int64_t { return NORM || pos < R ? pos : R - 1; };

  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = folx_wave_id();
  const int l32 = lane % 32;
  const int lh = lane / 32;

  // tile row 32 wave + l32 is Jacobian row p0 + l32 % PT of position r0 + (32 wave + l32) / PT
  const int64_t a_pos = inside(r0 + wave * PB + l32 / PT);
  const int64_t a_posg = PARTS ? a_pos / a.parts.group : 0;
  int a_row = p0 + l32 % PT;
  if (a_row >= P) a_row = P - 1;  // reaches accumulator rows that are neither stored nor summed
  const float* a_src = PARTS ? nullptr : a.jac + ((int64_t)a_row * R + a_pos) * K + 8 * lh;
  auto at = [&](int kt) __attribute__((always_inline)) -> const float* {
    if constexpr (PARTS) {
      // the part this chunk of K lies in: the same for the whole workgroup
      const int k0 = kt * BK;
      int sp = 0;
      while (sp + 1 < a.parts.n && k0 >= a.parts.kend[sp]) ++sp;
      const int32_t wd = a.parts.width[sp];
      return a.parts.jac[sp] + (int64_t)a_row * a.parts.pstride[sp] + (a.parts.bcast[sp] ? a_posg : a_pos) * wd +
             (k0 - (a.parts.kend[sp] - wd)) + 8 * lh;
    } else {
      return a_src + kt * BK;
    }
  };

  floatx16 acc[1][CB];
  // The per-walker pre-activation term is what the accumulators START from (the products are added to it): its
  // loads are in flight with the first chunk, where registers are plentiful, instead of in the epilogue.
  // Register r of a block <-> Jacobian row p0 + 4 (lane / 32) + 8 ((r / 4) % GB) + r % 4 of position (r / 4) / GB.
  auto start = [&](int j) __attribute__((always_inline)) {
    floatx16 v = folx_split::zeros();
    if constexpr (PARTS) {
      constexpr int GB = PT / 8;
      if (a.pre_jac != nullptr) {
        const int64_t pre_pstride = (R / a.pre_group) * N;
        const int gc = col0 + j * 32 + l32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int g = r / 4, b = g / GB;
          int prow = p0 + 4 * lh + 8 * (g % GB) + r % 4;
          if (prow >= P) prow = P - 1;  // rows past P of a ragged tile are neither stored nor summed
          v[r] = a.pre_jac[(int64_t)prow * pre_pstride + (inside(r0 + wave * PB + b) / a.pre_group) * N + (gc < N ? gc : N - 1)];
        }
      }
    }
    return v;
  };
  auto init = [&]() __attribute__((always_inline)) {
    if constexpr (!PARTS) {
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[0][j] = start(j);
    } else {
      floatx16 v[2];
      v[0] = start(0);
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if (j + 1 < CB) v[(j + 1) & 1] = start(j + 1);
        acc[0][j] = v[j & 1];
        asm volatile("" : "+v"(acc[0][j]));  // put together now: all blocks' values apart would take as many registers again
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // LayerNorm's row sums over the k that this lane half multiplies: sum t, sum xh t, sum t^2
  float sa = 0.0f, sb = 0.0f, s2 = 0.0f;
  auto seen = [&](int kt, const float4& u, const float4& v) __attribute__((always_inline)) {
    if constexpr (NORM) {
      const float4* xp = reinterpret_cast<const float4*>(&xhS[wave * K + kt * BK + 8 * lh]);
      const float4 xu = xp[0], xv = xp[1];
      sa += ((u.x + u.y) + (u.z + u.w)) + ((v.x + v.y) + (v.z + v.w));
      sb = fmaf(u.x, xu.x, fmaf(u.y, xu.y, fmaf(u.z, xu.z, fmaf(u.w, xu.w, sb))));
      sb = fmaf(v.x, xv.x, fmaf(v.y, xv.y, fmaf(v.z, xv.z, fmaf(v.w, xv.w, sb))));
      s2 = fmaf(u.x, u.x, fmaf(u.y, u.y, fmaf(u.z, u.z, fmaf(u.w, u.w, s2))));
      s2 = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, s2))));
    }
  };
  // what the epilogue needs per position and column
  auto meanwhile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int e = tid; e < RT * BN; e += Tile::NT) {
      int gc = col0 + e % BN;
      if (gc >= N) gc = N - 1;
      const float z = a.z[inside(r0 + e / BN) * N + gc];
      if constexpr (NORM) w2S[e] = z - a.c0[gc];
      if constexpr (ACT) {
        float f, d1, d2;
        act_eval_fused(a.act, z, a.prm, f, d1, d2);
        d1S[e] = d1;
      }
    }
    if constexpr (NORM) {
      if (tid < BN) w1S[tid] = a.w1[col0 + tid < N ? col0 + tid : N - 1];
      // xh of the tile's RT positions: RT * K consecutive floats
      const float4* src = reinterpret_cast<const float4*>(a.xhat + r0 * K);
      for (int e = tid; e < RT * K / 4; e += Tile::NT) reinterpret_cast<float4*>(xhS)[e] = src[e];
    }
  };
  const int32_t blocks = (N + 31) / 32;
  Tile::products(acc, ws0, ws1, a.pieces + (int64_t)(col0 / 32) * 1024, blocks, blocks - col0 / 32, K / BK, start, init, at, seen,
                 meanwhile);

  float rsv = 1.0f;
  if constexpr (NORM) {
    rsv = a.rs[r0 + wave];
    // the row sums go through LDS to the lanes that hold the rows' accumulators, inside the wavefront
    const float invK = 1.0f / (float)K;
    const bool pv = p0 + l32 < P;
    const float ta = sa + __shfl_xor(sa, 32, FOLX_WAVE);
    const float tb = sb + __shfl_xor(sb, 32, FOLX_WAVE);
    const float t2 = s2 + __shfl_xor(s2, 32, FOLX_WAVE);
    const float av = pv ? ta * invK : 0.0f;
    const float bv = pv ? tb * invK : 0.0f;
    const float qv = pv ? t2 * invK - av * av : 0.0f;
    if (lh == 0) st[wave * 32 + l32] = make_float2(av, bv);
    if (ct == 0) {  // the two scalar sums of the position
      float eb = bv * bv, eq = qv;
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) {
        eb += __shfl_xor(eb, off, FOLX_WAVE);
        eq += __shfl_xor(eq, off, FOLX_WAVE);
      }
      if (lane == 0) {
        float* o = a.sc + ((int64_t)pg * R + r0 + wave) * 2;
        o[0] = eb;
        o[1] = eq;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }

  // Register r of a block is tile row 8 (r / 4) + 4 (lane / 32) + r % 4 of the block, column
  // lane % 32: Jacobian row p0 + (that row) % PT of the block's position (that row) / PT.
  const int64_t pstride = R * N;  // floats between consecutive Jacobian rows
  const bool full_rows = (p0 + PT <= P) && (NORM || r0 + RT <= R);
  const int64_t pos = r0 + wave * PB;
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int gc = col0 + j * 32 + l32;
    const bool full_tile = full_rows && col0 + j * 32 + 32 <= N;
    float d1[PB];
#pragma unroll
    for (int b = 0; b < PB; ++b) d1[b] = ACT ? d1S[(wave * PB + b) * BN + j * 32 + l32] : 1.0f;
    float w1c = 0.0f, w2c = 0.0f;
    if constexpr (NORM) {
      w1c = w1S[j * 32 + l32];
      w2c = w2S[wave * BN + j * 32 + l32];
    }
    float* out = a.y_jac + ((int64_t)(p0 + 4 * lh) * R + pos) * N + gc;
    float ss[PB], s1 = 0.0f;
#pragma unroll
    for (int b = 0; b < PB; ++b) ss[b] = 0.0f;
    const float* resp = nullptr;
    if constexpr (PARTS) resp = a.res_jac ? a.res_jac + ((int64_t)(p0 + 4 * lh) * R + pos) * N + gc : nullptr;
    auto rows = [&](auto full, auto has_res, auto stream) __attribute__((always_inline)) {
      constexpr int GB = PT / 8;     // register groups per position
      constexpr bool FULL = decltype(full)::value, RES = decltype(has_res)::value;
      // What the epilogue reads from memory (the skip connection) is asked for one register group ahead
      // of its use: the stores of a group cannot be told apart from that array, so a load written after
      // them would wait for them to be issued, and every group would pay a round trip of its own.
      float rbuf[2][4];
      auto fetch = [&](int g, float (&rb)[4]) __attribute__((always_inline)) {
        const int b = g / GB;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int pl = 8 * (g % GB) + rr;
          const int64_t off = (int64_t)pl * pstride + (int64_t)b * N;
          const bool live = FULL || (p0 + 4 * lh + pl < P && gc < N && (NORM || pos + b < R));
          rb[rr] = 0.0f;
          if constexpr (RES) {
            if constexpr (FULL) rb[rr] = __builtin_nontemporal_load(resp + off);
            else if (live) rb[rr] = resp[off];
          }
        }
      };
      if constexpr (RES) fetch(0, rbuf[0]);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int b = g / GB;          // position of this group inside the block
        if constexpr (RES)
          if (g + 1 < 4) fetch(g + 1, rbuf[(g + 1) & 1]);
        float ap[4] = {0.0f, 0.0f, 0.0f, 0.0f}, bp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (NORM) {
          const float4* sp = reinterpret_cast<const float4*>(st + wave * 32 + 8 * g + 4 * lh);
          const float4 u0 = sp[0], u1 = sp[1];
          ap[0] = u0.x; bp[0] = u0.y; ap[1] = u0.z; bp[1] = u0.w;
          ap[2] = u1.x; bp[2] = u1.y; ap[3] = u1.z; bp[3] = u1.w;
        }
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int pl = 8 * (g % GB) + rr;
          float v = acc[0][j][4 * g + rr];
          if constexpr (NORM) {
            v = fmaf(-ap[rr], w1c, v);
            s1 = fmaf(bp[rr], v, s1);
            v = fmaf(-bp[rr], w2c, v) * rsv;
          }
          const int64_t off = (int64_t)pl * pstride + (int64_t)b * N;
          float* o = out + off;
          if constexpr (FULL) {
            if constexpr (ACT) ss[b] = fmaf(v, v, ss[b]);
            float w = d1[b] * v;
            if constexpr (RES) w += rbuf[g & 1][rr];
            if constexpr (decltype(stream)::value) __builtin_nontemporal_store(w, o);
            else *o = w;
          } else if (p0 + 4 * lh + pl < P && (NORM || pos + b < R)) {
            if constexpr (ACT) ss[b] = fmaf(v, v, ss[b]);
            if (gc < N) *o = d1[b] * v + (RES ? rbuf[g & 1][rr] : 0.0f);
          }
        }
      }
    };
    // (rows that do not end on a line: see store_tile in dense.hip)
    auto forms = [&](auto has_res) __attribute__((always_inline)) {
      if (!full_tile) rows(std::false_type{}, has_res, std::false_type{});
      else if (N % 32 == 0) rows(std::true_type{}, has_res, std::true_type{});
      else rows(std::true_type{}, has_res, std::false_type{});
    };
    if (PARTS && resp != nullptr) forms(std::true_type{});
    else forms(std::false_type{});
    const int64_t so = ((int64_t)pg * R + pos) * N + gc;
    if constexpr (ACT) {
#pragma unroll
      for (int b = 0; b < PB; ++b) {
        const float t = ss[b] + __shfl_xor(ss[b], 32, FOLX_WAVE);
        if (lh == 0 && gc < N && (NORM || pos + b < R)) a.ss[so + (int64_t)b * N] = t;
      }
    }
    if constexpr (NORM) {
      s1 += __shfl_xor(s1, 32, FOLX_WAVE);
      if (lh == 0 && gc < N) a.s1[so] = s1;
    }
  }
}

// Finishes the x and lap rows.  On entry y holds z and y_lap the part of zl that is linear in
// the input's lap row (what launch 2 left there).  One float4 per thread.
template <bool NORM, bool ACT>
__global__ __launch_bounds__(256) void wide_pieces_finish(float* __restrict__ y, float* __restrict__ y_lap,
                                                         const float* __restrict__ ss, const float* __restrict__ s1,
                                                         const float* __restrict__ sc, const float* __restrict__ rs,
                                                         const float* __restrict__ c0, int64_t S4, int64_t R,
                                                         int32_t N, int32_t PG, int32_t act, float prm,
                                                         const float* __restrict__ res,
                                                         const float* __restrict__ res_lap) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= S4) return;
  const float4 z = reinterpret_cast<const float4*>(y)[i];
  float4 zl = reinterpret_cast<const float4*>(y_lap)[i];
  if constexpr (NORM) {
    const int64_t pos = i / (N / 4);
    const int32_t n = (int32_t)(i % (N / 4)) * 4;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float eb = 0.0f, eq = 0.0f;
    for (int g = 0; g < PG; ++g) {
      const float4 t = reinterpret_cast<const float4*>(s1)[(int64_t)g * S4 + i];
      v.x += t.x; v.y += t.y; v.z += t.z; v.w += t.w;
      eb += sc[((int64_t)g * R + pos) * 2];
      eq += sc[((int64_t)g * R + pos) * 2 + 1];
    }
    const float r = rs[pos];
    const float r2 = r * r, e = 3.0f * eb - eq;
    zl.x += r2 * fmaf(z.x - c0[n], e, -2.0f * v.x);
    zl.y += r2 * fmaf(z.y - c0[n + 1], e, -2.0f * v.y);
    zl.z += r2 * fmaf(z.z - c0[n + 2], e, -2.0f * v.z);
    zl.w += r2 * fmaf(z.w - c0[n + 3], e, -2.0f * v.w);
  }
  if constexpr (ACT) {
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int g = 0; g < PG; ++g) {
      const float4 t = reinterpret_cast<const float4*>(ss)[(int64_t)g * S4 + i];
      s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
    }
    float4 f;
    float d1, d2;
    act_eval_fused(act, z.x, prm, f.x, d1, d2); zl.x = fmaf(d1, zl.x, d2 * s.x);
    act_eval_fused(act, z.y, prm, f.y, d1, d2); zl.y = fmaf(d1, zl.y, d2 * s.y);
    act_eval_fused(act, z.z, prm, f.z, d1, d2); zl.z = fmaf(d1, zl.z, d2 * s.z);
    act_eval_fused(act, z.w, prm, f.w, d1, d2); zl.w = fmaf(d1, zl.w, d2 * s.w);
    if (res) {
      const float4 r = reinterpret_cast<const float4*>(res)[i];
      f.x += r.x; f.y += r.y; f.z += r.z; f.w += r.w;
    }
    reinterpret_cast<float4*>(y)[i] = f;
  }
  if (res_lap) {
    const float4 r = reinterpret_cast<const float4*>(res_lap)[i];
    zl.x += r.x; zl.y += r.y; zl.z += r.z; zl.w += r.w;
  }
  reinterpret_cast<float4*>(y_lap)[i] = zl;
}

// The pieces of Wg = diag(gamma) W and per column w1 = 1^T Wg, c0 = bias + beta @ W.  A block takes 16 columns; its 16 groups of
// 16 lanes split the octets of K, and the partial sums meet within a wavefront first.
constexpr int FOLD_COLS = 16;

__device__ __forceinline__ void norm_fold(const float* __restrict__ W, const float* __restrict__ bias,
                                          const float* __restrict__ gamma, const float* __restrict__ beta,
                                          char* __restrict__ pieces, float* __restrict__ w1, float* __restrict__ c0, int32_t K,
                                          int32_t N, int block) {
  __shared__ float ps[4][FOLD_COLS], pc[4][FOLD_COLS];
  const int c = threadIdx.x % FOLD_COLS, sl = threadIdx.x / FOLD_COLS;
  const int n = block * FOLD_COLS + c;
  float s = 0.0f, cc = 0.0f;
  for (int octet = sl; octet < K / 8; octet += 16) {
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = n < N ? W[(int64_t)(octet * 8 + e) * N + n] : 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (beta) cc = fmaf(beta[octet * 8 + e], w[e], cc);
      if (gamma) w[e] *= gamma[octet * 8 + e];
      s += w[e];
    }
    folx_split::store_octet(w, pieces, octet, n, (N + 31) / 32);
  }
#pragma unroll
  for (int off = 32; off >= 16; off /= 2) {
    s += __shfl_xor(s, off, FOLX_WAVE);
    cc += __shfl_xor(cc, off, FOLX_WAVE);
  }
  if (sl % 4 == 0) { ps[sl / 4][c] = s; pc[sl / 4][c] = cc; }
  __syncthreads();
  if (sl == 0 && n < N) {
    w1[n] = (ps[0][c] + ps[1][c]) + (ps[2][c] + ps[3][c]);
    c0[n] = (bias ? bias[n] : 0.0f) + ((pc[0][c] + pc[1][c]) + (pc[2][c] + pc[3][c]));
  }
}

// One wavefront per position: xh, rs and, before gamma, the part of LN's lap row that is linear in the
// input's lap row, rs (lap - mean(lap) - xh mean(xh lap)).  K <= 512: two float4 per lane.
__device__ __forceinline__ void norm_rows(const float* __restrict__ x, const float* __restrict__ lap, float* __restrict__ xhat,
                                          float* __restrict__ rs, float* __restrict__ nlap, int64_t R, int32_t K, float eps,
                                          int64_t block) {
  const int lane = threadIdx.x % 64;
  const int64_t pos = block * 4 + threadIdx.x / 64;
  if (pos >= R) return;
  auto wsum = [](float v) __attribute__((always_inline)) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, FOLX_WAVE);
    return v;
  };
  const int nv = K / 4;
  const float invK = 1.0f / (float)K;
  float4 xv[2], lv[2];
  float s = 0.0f, sl = 0.0f;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int e = lane + 64 * c;
    xv[c] = lv[c] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (e < nv) {
      xv[c] = reinterpret_cast<const float4*>(x + pos * K)[e];
      lv[c] = reinterpret_cast<const float4*>(lap + pos * K)[e];
    }
    s += (xv[c].x + xv[c].y) + (xv[c].z + xv[c].w);
    sl += (lv[c].x + lv[c].y) + (lv[c].z + lv[c].w);
  }
  const float mean = wsum(s) * invK;
  const float aL = wsum(sl) * invK;
  float sv = 0.0f;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    if (lane + 64 * c < nv) {
      xv[c].x -= mean; xv[c].y -= mean; xv[c].z -= mean; xv[c].w -= mean;
      sv += xv[c].x * xv[c].x + xv[c].y * xv[c].y + xv[c].z * xv[c].z + xv[c].w * xv[c].w;
    }
  }
  const float r = 1.0f / sqrtf(wsum(sv) * invK + eps);
  float sbl = 0.0f;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    xv[c].x *= r; xv[c].y *= r; xv[c].z *= r; xv[c].w *= r;
    sbl += xv[c].x * lv[c].x + xv[c].y * lv[c].y + xv[c].z * lv[c].z + xv[c].w * lv[c].w;
  }
  const float bL = wsum(sbl) * invK;
  if (lane == 0) rs[pos] = r;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int e = lane + 64 * c;
    if (e < nv) {
      reinterpret_cast<float4*>(xhat + pos * K)[e] = xv[c];
      reinterpret_cast<float4*>(nlap + pos * K)[e] =
          make_float4(r * (lv[c].x - aL - bL * xv[c].x), r * (lv[c].y - aL - bL * xv[c].y),
                      r * (lv[c].z - aL - bL * xv[c].z), r * (lv[c].w - aL - bL * xv[c].w));
    }
  }
}

// Both in one launch, the blocks of the weights first: neither reads what the other writes.  K = N = 256: 16.5 us for the weights
// (64 columns a block, 16 requests in a row each) and 4.9 us for the rows of 640 positions, each its own launch, became 6 us.
// The fused form is the one for any number of positions, also where LayerNorm and the plain product would be faster (P R < 30 000: 1.4 times
// in the mean over 77 sizes): the two round differently, and a
// walker's Jacobian then depended on how many walkers a call has, by up to 1.5e-3 of it behind a determinant of 20 electrons.
__global__ __launch_bounds__(256) void norm_prepare_kernel(const float* x, const float* lap, const float* W, const float* bias,
                                                           const float* gamma, const float* beta, float* xhat, float* rs,
                                                           float* nlap, char* pieces, float* w1, float* c0, int64_t R,
                                                           int32_t K, int32_t N, float eps) {
  const int fold = (N + 31) / 32 * (32 / FOLD_COLS);
  if ((int)blockIdx.x < fold) norm_fold(W, bias, gamma, beta, pieces, w1, c0, K, N, (int)blockIdx.x);
  else norm_rows(x, lap, xhat, rs, nlap, R, K, eps, (int64_t)blockIdx.x - fold);
}

// y[r][c] += pre[r / group][c], y_lap likewise: the per-walker pre-activation term on the x and lap
// rows (one float4 per thread).
__global__ __launch_bounds__(256) void wide_add_pre_kernel(float* __restrict__ y, float* __restrict__ y_lap,
                                                           const float* __restrict__ pre,
                                                           const float* __restrict__ pre_lap, int64_t S4, int32_t N4,
                                                           int64_t group) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= S4) return;
  const int64_t src = (i / N4 / group) * N4 + i % N4;
  float4 a = reinterpret_cast<float4*>(y)[i], b = reinterpret_cast<float4*>(y_lap)[i];
  const float4 p = reinterpret_cast<const float4*>(pre)[src], q = reinterpret_cast<const float4*>(pre_lap)[src];
  a.x += p.x; a.y += p.y; a.z += p.z; a.w += p.w;
  b.x += q.x; b.y += q.y; b.z += q.z; b.w += q.w;
  reinterpret_cast<float4*>(y)[i] = a;
  reinterpret_cast<float4*>(y_lap)[i] = b;
}

// Shapes the path takes, launch sizes and the carve-up of the workspace (offsets in floats,
// every part a multiple of 4 floats).
struct WidePlan {
  int64_t row_tiles, pos_tiles, blocks, ws_bytes, asked_bytes;
  int64_t o_ss, o_s1, o_sc, o_xhat, o_rs, o_nlap, o_pieces, o_w1, o_c0;
  int32_t PG, PT, CB, col_tiles;
};

// The forms of the fused layers (PiecesRates, from the same 520 layers, 107 of them behind LayerNorm; 7 % rms): groups of 8,
// 16 and 32 Jacobian rows, tiles of 8 and 4 blocks of columns.  Their launches besides the products are in `launch`.
constexpr PiecesRates WIDE_ACT[3][2] = {{{8, 2, 22.3, 0.062, 0.0977, 8.75, 0.164, 0.76}, {4, 3, 21.2, 0.076, 0.0833, 3.43, 0.161, 0.41}},
                                        {{8, 2, 19.7, 0.070, 0.1003, 7.56, 0.134, 0.68}, {4, 3, 18.4, 0.074, 0.0903, 3.47, 0.130, 0.41}},
                                        {{8, 2, 17.9, 0.074, 0.1041, 6.27, 0.120, 0.63}, {4, 3, 16.6, 0.075, 0.0897, 3.78, 0.120, 0.42}}};
constexpr PiecesRates WIDE_NORM[2] = {{8, 2, 28.4, 0.033, 0.0990, 2.62, 0.186, 0.72}, {4, 3, 25.6, 0.041, 0.0817, 1.74, 0.193, 0.51}};

double wide_time(const PiecesRates& c, int64_t R, int32_t P, int32_t K, int32_t N, int PT) {
  const int64_t groups = (P + PT - 1) / PT, tiles = (R + BM / PT - 1) / (BM / PT) * groups;
  return folx_pieces_time(c, tiles * ((N + 32 * c.blocks - 1) / (32 * c.blocks)), K,
                          4e-6 * (double)R * ((double)P * (K + N) + (double)N * (double)(groups + 6)));
}

// The form of least estimated time: 1.005 times the fastest one's in the mean for the activation alone, 1.003 behind LayerNorm
// (whose row sums need groups of 32).
double wide_form(bool norm, int64_t R, int32_t P, int32_t K, int32_t N, int32_t& PT, int32_t& CB) {
  double least = -1.0;
  for (int g = 0; g < 3; ++g) {
    if (norm && g < 2) continue;
    for (const PiecesRates& c : norm ? WIDE_NORM : WIDE_ACT[g]) {
      const double t = wide_time(c, R, P, K, N, 8 << g);
      if (least < 0.0 || t < least) { least = t; PT = 8 << g; CB = c.blocks; }
    }
  }
  return least;
}

// The plain product over K features and the activation after it
double plain_time(int64_t R, int32_t P, int32_t K, int32_t N) {
  const int64_t rows[3] = {R, P * R, R};
  double t;
  folx_pieces_columns(rows, K, N, &t);
  return t + 3.0 + 0.155 * 8e-6 * (double)R * N * (P + 2);
}

bool plan_wide(int64_t R, int32_t P, int32_t K, int32_t N, bool norm, bool act, WidePlan& pl) {
  if (R <= 0 || R % 4 != 0 || P < 1 || K < BK || K % BK != 0 || N <= 128 || N % 4 != 0) return false;
  if (norm && K > KMAX_NORM) return false;
  wide_form(norm, R, P, K, N, pl.PT, pl.CB);
  pl.PG = (P + pl.PT - 1) / pl.PT;
  pl.pos_tiles = (R + BM / pl.PT - 1) / (BM / pl.PT);
  pl.row_tiles = pl.pos_tiles * pl.PG;
  pl.col_tiles = (N + 32 * pl.CB - 1) / (32 * pl.CB);
  pl.blocks = (pl.row_tiles + NXCD - 1) / NXCD * NXCD * pl.col_tiles;
  if (pl.blocks > 0x7fffffffLL) return false;
  if (R * (int64_t)N / 4 / 256 + 1 > 0x7fffffffLL) return false;
  const int64_t slab = (int64_t)pl.PG * R * N;
  int64_t o = 0;
  auto take = [&](int64_t n) { const int64_t at = o; o += (n + 3) / 4 * 4; return at; };
  pl.o_ss = act ? take(slab) : 0;
  pl.o_pieces = take(folx_split::pieces_bytes(K, N) / 4);
  if (norm) {
    pl.o_s1 = take(slab);
    pl.o_sc = take((int64_t)pl.PG * R * 2);
    pl.o_xhat = take(R * (int64_t)K);
    pl.o_rs = take(R);
    pl.o_nlap = take(R * (int64_t)K);
    pl.o_w1 = take(N);
    pl.o_c0 = take(N);
  }
  pl.ws_bytes = o * 4;
  if (norm) {
    // What the query has always said: pieces of Wg and no copy of LN(x) take less than Wg and that copy, but for few
    // positions of many features.
    const int64_t asked = 4 * (o - folx_split::pieces_bytes(K, N) / 4 + (int64_t)K * N + R * (int64_t)K);
    pl.asked_bytes = asked;
    if (pl.ws_bytes < asked) pl.ws_bytes = asked;
  }
  return true;
}

template <bool NORM, bool ACT, int PT, bool PARTS = false>
int launch_wide(hipStream_t st, const WideParams& a, const WidePlan& pl, float* y, float* y_lap,
                const float* res = nullptr, const float* res_lap = nullptr) {
  const dim3 grid((unsigned)pl.blocks), block(256);
  auto launch = [&](auto apart) {
    constexpr bool APART = decltype(apart)::value;
    if (pl.CB == 8) wide_pieces_kernel<8, NORM, ACT, PT, PARTS, APART><<<grid, block, 0, st>>>(a);
    else wide_pieces_kernel<4, NORM, ACT, PT, PARTS, APART><<<grid, block, 0, st>>>(a);
  };
  if constexpr (NORM) {
    launch(std::false_type{});  // K <= KMAX_NORM
  } else {
    if (a.K > folx_split::APART_K) launch(std::true_type{});
    else launch(std::false_type{});
  }
  int rc = folx_launch_status();
  if (rc != FOLX_HIP_OK) return rc;
  const int64_t S4 = a.R * (int64_t)a.N / 4;
  wide_pieces_finish<NORM, ACT><<<dim3((unsigned)((S4 + 255) / 256)), dim3(256), 0, st>>>(
      y, y_lap, a.ss, a.s1, a.sc, a.rs, a.c0, S4, a.R, a.N, pl.PG, a.act, a.prm, res, res_lap);
  return folx_launch_status();
}

int run_wide(hipStream_t st, bool norm, int32_t act, float param, const float* x, const float* jac, const float* lap,
             const float* gamma, const float* beta, float eps, const float* W, const float* bias, float* y,
             float* y_jac, float* y_lap, int64_t R, int32_t P, int32_t K, int32_t N, void* workspace,
             int64_t workspace_bytes, const WideParts* parts = nullptr, const float* res = nullptr,
             const float* res_jac = nullptr, const float* res_lap = nullptr, const float* pre = nullptr,
             const float* pre_jac = nullptr, const float* pre_lap = nullptr, int64_t pre_group = 1) {
  const bool has_act = act >= 0;
  WidePlan pl;
  if ((has_act && !act_fused(act)) || !plan_wide(R, P, K, N, norm, has_act, pl)) return FOLX_HIP_ENOTSUP;
  if (!norm && !has_act) return FOLX_HIP_ENOTSUP;  // that is the plain dense rule
  if (parts && norm) return FOLX_HIP_ENOTSUP;
  if (!x || (!jac && !parts) || !lap || !W || !y || !y_jac || !y_lap) return FOLX_HIP_EINVAL;
  if (!folx_aligned16(jac) || !folx_aligned16(W) || !folx_aligned16(y) || !folx_aligned16(y_lap))
    return FOLX_HIP_ENOTSUP;
  if (norm && (!folx_aligned16(x) || !folx_aligned16(lap) || !folx_aligned16(gamma) || !folx_aligned16(beta)))
    return FOLX_HIP_ENOTSUP;
  if (!workspace || workspace_bytes < pl.ws_bytes || !folx_aligned16(workspace)) return FOLX_HIP_EINVAL;
  float* ws = (float*)workspace;
  WideParams a;
  a.jac = jac; a.pieces = (const char*)(ws + pl.o_pieces); a.z = y; a.y_jac = y_jac; a.res_jac = res_jac;
  a.pre_jac = pre_jac; a.pre_group = pre_group;
  a.xhat = nullptr; a.rs = nullptr; a.w1 = a.c0 = nullptr;
  a.ss = ws + pl.o_ss; a.s1 = nullptr; a.sc = nullptr;
  a.R = R; a.row_tiles = pl.row_tiles; a.pos_tiles = pl.pos_tiles;
  a.P = P; a.K = K; a.N = N; a.col_tiles = pl.col_tiles; a.act = act; a.prm = param;
  const float* in_x = x;
  const float* in_lap = lap;
  const float* in_bias = bias;
  if (norm) {
    const int64_t blocks = (N + 31) / 32 * (32 / FOLD_COLS) + (R + 3) / 4;
    if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
    norm_prepare_kernel<<<dim3((unsigned)blocks), dim3(256), 0, st>>>(
        x, lap, W, bias, gamma, beta, ws + pl.o_xhat, ws + pl.o_rs, ws + pl.o_nlap, (char*)(ws + pl.o_pieces), ws + pl.o_w1,
        ws + pl.o_c0, R, K, N, eps);
    const int rc = folx_launch_status();
    if (rc != FOLX_HIP_OK) return rc;
    a.xhat = ws + pl.o_xhat; a.rs = ws + pl.o_rs; a.w1 = ws + pl.o_w1; a.c0 = ws + pl.o_c0;
    a.s1 = ws + pl.o_s1; a.sc = ws + pl.o_sc;
    // LN(x) @ W + bias = xh @ Wg + c0
    in_x = a.xhat; in_lap = ws + pl.o_nlap; in_bias = a.c0;
  }
  // z and the linear part of zl: no Jacobian rows, no residual
  int rc = folx_dense_values(st, in_x, in_lap, norm ? nullptr : W, const_cast<char*>(a.pieces), in_bias, y, y_lap, R, K, N);
  if (rc != FOLX_HIP_OK) return rc;
  if (pre) {
    const int64_t S4 = R * (int64_t)N / 4;
    wide_add_pre_kernel<<<dim3((unsigned)((S4 + 255) / 256)), dim3(256), 0, st>>>(y, y_lap, pre, pre_lap, S4, N / 4,
                                                                              pre_group);
    rc = folx_launch_status();
    if (rc != FOLX_HIP_OK) return rc;
  }
  if (norm)
    return has_act ? launch_wide<true, true, 32>(st, a, pl, y, y_lap) : launch_wide<true, false, 32>(st, a, pl, y, y_lap);
  if (parts) {
    a.parts = *parts;
    return pl.PT == 8    ? launch_wide<false, true, 8, true>(st, a, pl, y, y_lap, res, res_lap)
           : pl.PT == 16 ? launch_wide<false, true, 16, true>(st, a, pl, y, y_lap, res, res_lap)
                         : launch_wide<false, true, 32, true>(st, a, pl, y, y_lap, res, res_lap);
  }
  return pl.PT == 8    ? launch_wide<false, true, 8>(st, a, pl, y, y_lap)
         : pl.PT == 16 ? launch_wide<false, true, 16>(st, a, pl, y, y_lap)
                       : launch_wide<false, true, 32>(st, a, pl, y, y_lap);
}

}  // namespace

int folx_wide_pieces_faster(int64_t R, int32_t P, int32_t K, int32_t N, int32_t plain) {
  WidePlan pl;
  if (!plan_wide(R, P, K, N, false, true, pl)) return FOLX_HIP_ENOTSUP;
  // An operand read in parts spares features, and rounds differently: where its tiles are well filled, for any number of positions.
  const int32_t base = R % 8 == 0 && (P + 15) / 16 * 16 < (P + 31) / 32 * 32 ? 16 : 32;
  if (plain > K && (P + base - 1) / base * base <= 1.125 * P) return 1;
  int32_t pt, cb;
  return wide_form(false, R, P, K, N, pt, cb) < plain_time(R, P, plain, N);
}

int64_t folx_wide_pieces_ws_bytes(int64_t R, int32_t P, int32_t K, int32_t N) {
  WidePlan pl;
  return plan_wide(R, P, K, N, false, true, pl) ? pl.ws_bytes : FOLX_HIP_ENOTSUP;
}

int folx_wide_pieces(hipStream_t st, int32_t act, float param, const float* x, const float* jac, const float* lap,
                     const FolxWideParts* parts, const float* W, const float* bias, const float* res, const float* res_jac,
                     const float* res_lap, const float* pre, const float* pre_jac, const float* pre_lap, int64_t pre_group,
                     float* y, float* y_jac, float* y_lap, int64_t R, int32_t P, int32_t K, int32_t N, void* workspace,
                     int64_t workspace_bytes) {
  return run_wide(st, false, act, param, x, jac, lap, nullptr, nullptr, 0.0f, W, bias, y, y_jac, y_lap, R, P, K, N, workspace,
                  workspace_bytes, parts, res, res_jac, res_lap, pre, pre_jac, pre_lap, pre_group);
}

extern "C" int64_t folx_hip_norm_dense_workspace_bytes(int64_t R, int32_t P, int32_t K, int32_t N, int32_t act) {
  if (R < 0 || P < 0 || K <= 0 || N <= 0) return FOLX_HIP_EINVAL;
  WidePlan pl;
  if ((act >= 0 && !act_fused(act)) || !plan_wide(R, P, K, N, true, act >= 0, pl)) return FOLX_HIP_ENOTSUP;
  return pl.ws_bytes;
}

extern "C" int folx_hip_norm_dense_fwdlap(void* stream, int32_t act, float param, const float* x, const float* jac,
                                          const float* lap, const float* gamma, const float* beta, float eps,
                                          const float* W, const float* bias, float* y, float* y_jac, float* y_lap,
                                          int64_t R, int32_t P, int32_t K, int32_t N, void* workspace,
                                          int64_t workspace_bytes) {
  if (R < 0 || P < 0 || K <= 0 || N <= 0) return FOLX_HIP_EINVAL;
  return run_wide((hipStream_t)stream, true, act, param, x, jac, lap, gamma, beta, eps, W, bias, y, y_jac, y_lap, R, P,
                  K, N, workspace, workspace_bytes);
}

// ---- folx_hip_norm_dense_fwdlap on the library's own scratch memory -------------------------
//
// For callers that cannot bring a workspace because they cannot allocate one (code under HIP
// graph capture, tight serving loops).  The workspace of run_wide() is a file-scope device
// array; every GPU the library runs on holds its own copy of it, at its own address, until the
// process ends.  In host code the array's name is only a handle of the symbol, so the device
// address is asked for once per device (hipGetSymbolAddress, with that device current) and
// kept; everything below uses the pointer, never the name.
namespace {

// with room for the pieces of Wg where they are larger than Wg and a copy of LN(x): 2 K N - 4 R K bytes and the padded columns
constexpr int64_t SCRATCH_BYTES = FOLX_HIP_STATIC_SCRATCH_BYTES + (33ll << 20);
constexpr int MAX_DEVICES = 64;

}  // namespace

static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

void* g_scratch_ptr[MAX_DEVICES];  // device address of `scratch` on each device, once known
std::mutex g_scratch_mutex;

// Address of this device's copy of `scratch`; nullptr when the runtime refuses.
void* scratch_of_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int folx_hip_norm_dense_static_fwdlap(void* stream, int32_t act, float param, const float* x,
                                                 const float* jac, const float* lap, const float* gamma,
                                                 const float* beta, float eps, const float* W, const float* bias,
                                                 float* y, float* y_jac, float* y_lap, int64_t R, int32_t P,
                                                 int32_t K, int32_t N) {
  if (R < 0 || P < 0 || K <= 0 || N <= 0) return FOLX_HIP_EINVAL;
  WidePlan pl;
  if ((act >= 0 && !act_fused(act)) || !plan_wide(R, P, K, N, true, act >= 0, pl)) return FOLX_HIP_ENOTSUP;
  if (pl.asked_bytes > FOLX_HIP_STATIC_SCRATCH_BYTES || pl.ws_bytes > SCRATCH_BYTES) return FOLX_HIP_ESCRATCH;
  void* ptr = scratch_of_current_device();
  if (!ptr) return FOLX_HIP_ELAUNCH;
  // Nothing in the workspace has to start at zero: every launch of run_wide() writes the part
  // it owns (folded weights, per-position rows, one slab of sums per group of Jacobian rows)
  // in full before a later launch on the same stream reads it.
  return run_wide((hipStream_t)stream, true, act, param, x, jac, lap, gamma, beta, eps, W, bias, y, y_jac, y_lap, R, P,
                  K, N, ptr, SCRATCH_BYTES);
}
