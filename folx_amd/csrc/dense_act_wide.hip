// Wide dense layer (N > 128, K a multiple of 16) with the activation folded into the GEMM over the Jacobian rows, so that the
// pre-activation Jacobian does not go through HBM: y = f(x @ W + bias), for callers whose workspace holds the sums only (with room
// for W's pieces as well: wide_pieces.hip, which explains the tiles).  With z = x @ W + bias, zj[p] and zl the pre-activation
// triplet, y = f(z),  yj[p] = f'(z) zj[p],  yl = f'(z) zl + f''(z) sum_p zj[p]^2.
//
// Launches on the caller's stream:
//  1. the plain dense kernel on the x and lap rows only (2 R of the (P + 2) R rows): z goes to
//     y, zl to y_lap;
//  2. the Jacobian GEMM below, whose 128-row tiles are cut ACROSS Jacobian rows: a tile holds
//     4 consecutive positions x 32 consecutive p (or 8 x 16, 16 x 8), ordered position-major, so that f'(z) of an accumulator
//     block is one value per lane and position, and the sums over p inside a block stay inside the
//     wavefront.  They go to the workspace, one (R, N) slab per group of Jacobian rows;
//  3. a short elementwise kernel that finishes y and y_lap, adding the slabs in a fixed order.
//
// It also reads a CONCATENATED operand part by part (a chunk of 16 features lies in
// exactly one part; a part may hold one row per walker that all of the walker's positions
// share) and adds a skip connection in its epilogue, so that a layer fed by
// [own features, per-walker means, ...] forms neither the broadcasts nor the concatenation.
//
// The main loop is the one of the dense kernel: K in chunks of 16 through double-buffered LDS
// tiles filled by global_load_lds_dwordx4, a 128 x 256 tile on 8 wavefronts of 64 x 64,
// v_mfma_f32_32x32x2_f32 with the k order inside a group of 8 permuted to fit 128-bit reads
// (lane l, register j of group t <-> k = 8 t + 4 (l / 32) + j), piece c of an A row stored at
// slot c ^ ((row / 2) % 4).  Only the address a lane asks for differs: tile row m is
// Jacobian row p0 + m % 32 of position r0 + m / 32.
#include <algorithm>
#include <type_traits>

#include "activations.h"
#include "dense_act_wide.h"
#include "dense_tiles.h"
#include "split_bf16.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

#define FOLX_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define FOLX_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

constexpr int BK = 16;
constexpr int BM = 128, BN = 256, WM = 2, WN = 4;
constexpr int NT = 64 * WM * WN;
constexpr int WROWS = BM / WM, WCOLS = BN / WN;
constexpr int TM = WROWS / 32, TN = WCOLS / 32;
constexpr int TG = BK / 8;
constexpr int NXCD = 8;
constexpr int A_V4 = BM * BK / 4, W_V4 = BK * BN / 4;
constexpr int A_LD = A_V4 / NT, W_LD = W_V4 / NT;
static_assert(A_V4 % NT == 0 && W_V4 % NT == 0, "every thread loads the same number of pieces");

using WideParts = FolxWideParts;
constexpr int MAX_PARTS = FOLX_MAX_PARTS;

struct WideParams {
  const float* jac;
  const float* W;
  const float* z;    // pre-activation values (R, N), bias included
  float* y_jac;
  const float* res_jac;  // optional (P, R, N) added to the activated Jacobian rows     PARTS instances only
  const float* pre_jac;  // optional (P, R / pre_group, N) added to the PRE-activation Jacobian rows: position r takes
  int64_t pre_group;     // row r / pre_group (a per-walker term shared by the walker's positions)   PARTS instances only
  float* ss;         // (PG, R, N) sums of zj^2 per group of PT Jacobian rows     activation only
  int64_t R, row_tiles, pos_tiles;
  int32_t P, K, N, col_tiles, act;
  float prm;
  WideParts parts;   // PARTS instances only (jac unused then)
};

// PT = Jacobian rows of a tile: 32 (4 positions per tile, one per accumulator block), or 16 for
// the activation alone (8 positions per tile, two per block: registers 0-7 of a block belong
// to the first, 8-15 to the second), or 8 (four per block): fewer empty rows (P = 21 fills 24 instead of 32, P = 39 fills 40
// instead of 48 or 64) for more epilogue work per row (act_group).  A 7-electron FermiNet-style step of
// 512 walkers, whose layers went unfused with 832 instead of 320 contracted features: 2.58 -> 1.48 ms.  The activation's tiles may
// hold more positions than are left: those past R read position R - 1 and are neither stored nor summed.
// SPLIT: the products on the bf16 matrix pipe from operands split into three bf16 pieces, with
// the loop of dense_split_kernel: A and W chunks come through registers and every element is
// split once per workgroup on its way into LDS (A stage [piece][g][row][8 bf16], W stage
// [piece][g][kp][col] dwords).  A concatenated operand (PARTS) is staged the same way, the part of a chunk
// and the address inside it found per chunk as in the direct-to-LDS form.
template <int PT, bool PARTS, bool SPLIT>
__global__ __launch_bounds__(NT, 4) void dense_wide_kernel(WideParams a) {
  static_assert(!PARTS || A_LD == 1, "one A piece per thread");
  constexpr int A_PLANE = 2 * BM * 16;     // SPLIT: bytes of one piece of an A chunk
  constexpr int W_PLANE = 2 * 4 * BN * 4;  //        and of a W chunk
  constexpr int RT = BM / PT;  // positions of a tile
  constexpr int PB = 32 / PT;  // positions of a 32-row accumulator block
  static_assert(PT == 32 || PT == 16 || PT == 8, "one, two or four positions per block");
  __shared__ __attribute__((aligned(16))) float As0[SPLIT ? 3 * A_PLANE / 4 : BM * BK];
  __shared__ __attribute__((aligned(16))) float As1[SPLIT ? 3 * A_PLANE / 4 : BM * BK];
  __shared__ __attribute__((aligned(16))) float Ws0[SPLIT ? 3 * W_PLANE / 4 : BK * BN];
  __shared__ __attribute__((aligned(16))) float Ws1[SPLIT ? 3 * W_PLANE / 4 : BK * BN];

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
  auto inside = [&](int64_t pos) __attribute__((always_inline)) -> int64_t { return pos < R ? pos : R - 1; };

  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wrow = wave / WN;
  const int wr = wrow * WROWS;
  const int wc = (wave % WN) * WCOLS;
  const int l32 = lane % 32;
  const int lh = lane / 32;

  const float* a_p[A_LD];
  const float* w_p[W_LD];
  int64_t a_pos = 0, a_posg = 0;  // PARTS: this thread's position, and its row in a broadcast part
  int32_t a_row = 0, a_kc = 0;    //        its Jacobian row and 16-byte piece
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    const int idx = tid + NT * i;
    const int m = idx / 4, c = idx % 4;
    const int kc = c ^ ((m / 2) % 4);
    int p = p0 + m % PT;
    if (p >= P) p = P - 1;  // reaches accumulator rows that are neither stored nor summed
    if constexpr (PARTS) {
      a_pos = inside(r0 + m / PT);
      a_posg = a_pos / a.parts.group;
      a_row = p;
      a_kc = kc * 4;
      a_p[i] = nullptr;
    } else {
      a_p[i] = a.jac + ((int64_t)p * R + inside(r0 + m / PT)) * K + kc * 4;  // tile row m: position m / PT, row m % PT
    }
  }
#pragma unroll
  for (int i = 0; i < W_LD; ++i) {
    const int idx = tid + NT * i;
    const int k = (idx / (BN / 4)) % BK;
    int n = col0 + (idx % (BN / 4)) * 4;
    if (n > N - 4) n = N - 4;
    w_p[i] = a.W + (int64_t)k * N + n;
  }
  auto issue = [&](int kt, float* as, float* ws) __attribute__((always_inline)) {
    if constexpr (PARTS) {
      // the part this chunk of K lies in: the same for the whole workgroup
      const int k0 = kt * BK;
      int sp = 0;
      while (sp + 1 < a.parts.n && k0 >= a.parts.kend[sp]) ++sp;
      const int32_t wd = a.parts.width[sp];
      const float* src = a.parts.jac[sp] + (int64_t)a_row * a.parts.pstride[sp] +
                         (a.parts.bcast[sp] ? a_posg : a_pos) * wd + (k0 - (a.parts.kend[sp] - wd)) + a_kc;
      __builtin_amdgcn_global_load_lds(FOLX_GPTR(src), FOLX_LPTR(&as[(wave * 64) * 4]), 16, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < A_LD; ++i)
        __builtin_amdgcn_global_load_lds(FOLX_GPTR(a_p[i] + kt * BK), FOLX_LPTR(&as[(wave * 64 + NT * i) * 4]), 16,
                                         0, 0);
    }
#pragma unroll
    for (int i = 0; i < W_LD; ++i)
      __builtin_amdgcn_global_load_lds(FOLX_GPTR(w_p[i] + (int64_t)kt * BK * N),
                                       FOLX_LPTR(&ws[(wave * 64 + NT * i) * 4]), 16, 0, 0);
  };

  // z is asked for first, then the first chunk, and f' is evaluated while the chunk is on its way.
  float dr[TM][TN][PB];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      int gc = col0 + wc + j * 32 + l32;
      if (gc >= N) gc = N - 1;
#pragma unroll
      for (int b = 0; b < PB; ++b) dr[i][j][b] = a.z[inside(r0 + (wrow * TM + i) * PB + b) * N + gc];
    }
  // SPLIT staging: thread t has k quarter t % 4 of tile row t / 4; wavefront w has rows 2 w and
  // 2 w + 1 of the W chunk, lane l their columns 4 l .. 4 l + 3
  const float* sa_src = nullptr;
  const float* sw_src = nullptr;
  int sa_dst = 0, sw_dst = 0;
  float4 ra = make_float4(0.f, 0.f, 0.f, 0.f), rw0 = ra, rw1 = ra;
  if constexpr (SPLIT) {
    const int m = tid / 4, q = tid % 4;
    int p = p0 + m % PT;
    if (p >= P) p = P - 1;
    if constexpr (PARTS) {  // the part and the address inside it are found per chunk
      a_pos = inside(r0 + m / PT);
      a_posg = a_pos / a.parts.group;
      a_row = p;
      a_kc = q * 4;
    } else {
      sa_src = a.jac + ((int64_t)p * R + inside(r0 + m / PT)) * K + q * 4;
    }
    sa_dst = ((q / 2) * BM + m) * 16 + (q % 2) * 8;
    int wn = col0 + lane * 4;
    if (wn > N - 4) wn = N - 4;
    sw_src = a.W + (int64_t)(2 * wave) * N + wn;
    sw_dst = (wave * BN + lane * 4) * 4;
  }
  auto fetch = [&](int kt) __attribute__((always_inline)) {
    if constexpr (PARTS) {
      const int k0 = kt * BK;
      int sp = 0;
      while (sp + 1 < a.parts.n && k0 >= a.parts.kend[sp]) ++sp;
      const int32_t wd = a.parts.width[sp];
      ra = *reinterpret_cast<const float4*>(a.parts.jac[sp] + (int64_t)a_row * a.parts.pstride[sp] +
                                            (a.parts.bcast[sp] ? a_posg : a_pos) * wd + (k0 - (a.parts.kend[sp] - wd)) + a_kc);
    } else {
      ra = *reinterpret_cast<const float4*>(sa_src + kt * BK);  // plain: the line's other half follows one chunk later
    }
    rw0 = *reinterpret_cast<const float4*>(sw_src + (int64_t)kt * BK * N);
    rw1 = *reinterpret_cast<const float4*>(sw_src + (int64_t)kt * BK * N + N);
  };
  if constexpr (SPLIT) fetch(0);
  else issue(0, As0, Ws0);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int b = 0; b < PB; ++b) {
        float f, d1, d2;
        act_eval_fused(a.act, dr[i][j][b], a.prm, f, d1, d2);
        dr[i][j][b] = d1;
      }
  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  if constexpr (PARTS) {
    // The per-walker pre-activation term is what the accumulators START from (the products are added to it): its
    // loads are in flight with the first chunk, where registers are plentiful, instead of in the epilogue.
    // Register r of a block <-> Jacobian row p0 + 4 (lane / 32) + 8 ((r / 4) % GB) + r % 4 of position (r / 4) / GB.
    if (a.pre_jac) {
      constexpr int GB = PT / 8;
      const int64_t pre_pstride = (R / a.pre_group) * N;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          int gc = col0 + wc + j * 32 + l32;
          if (gc >= N) gc = N - 1;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int g = r / 4, b = g / GB;
            int prow = p0 + 4 * lh + 8 * (g % GB) + r % 4;
            if (prow >= P) prow = P - 1;  // rows past P of a ragged tile are neither stored nor summed
            const int64_t pos = inside(r0 + (wrow * TM + i) * PB + b);
            acc[i][j][r] = a.pre_jac[(int64_t)prow * pre_pstride + (pos / a.pre_group) * N + gc];
          }
        }
    }
  }
  const int sw = (l32 / 2) % 4;
  auto compute = [&](const float* as, const float* ws) __attribute__((always_inline)) {
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
      float4 a4[TM];
      float b[TN][4];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        a4[i] = *reinterpret_cast<const float4*>(&as[(wr + i * 32 + l32) * BK + (((tg * 2 + lh) ^ sw) * 4)]);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) b[j][q] = ws[(tg * 8 + lh * 4 + q) * BN + wc + j * 32 + l32];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const float av = q == 0 ? a4[i].x : (q == 1 ? a4[i].y : (q == 2 ? a4[i].z : a4[i].w));
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, b[j][q], acc[i][j], 0, 0, 0);
        }
      }
    }
  };

  const int KT = K / BK;
  if constexpr (SPLIT) {
    using namespace folx_split;
    // chunk kt of this thread's registers into a stage
    auto put = [&](int kt, float* asf, float* wsf) __attribute__((always_inline)) {
      char* as = reinterpret_cast<char*>(asf);
      char* ws = reinterpret_cast<char*>(wsf);
      unsigned p1a, p2a, p3a, p1b, p2b, p3b;
      split_pair(ra.x, ra.y, p1a, p2a, p3a);
      split_pair(ra.z, ra.w, p1b, p2b, p3b);
      uint2v q;
      q[0] = p1a; q[1] = p1b; *reinterpret_cast<uint2v*>(as + sa_dst) = q;
      q[0] = p2a; q[1] = p2b; *reinterpret_cast<uint2v*>(as + A_PLANE + sa_dst) = q;
      q[0] = p3a; q[1] = p3b; *reinterpret_cast<uint2v*>(as + 2 * A_PLANE + sa_dst) = q;
      unsigned a1[4], a2[4], a3[4];
      split_pair(rw0.x, rw1.x, a1[0], a2[0], a3[0]);
      split_pair(rw0.y, rw1.y, a1[1], a2[1], a3[1]);
      split_pair(rw0.z, rw1.z, a1[2], a2[2], a3[2]);
      split_pair(rw0.w, rw1.w, a1[3], a2[3], a3[3]);
      uint4v q1, q2, q3;
#pragma unroll
      for (int c = 0; c < 4; ++c) { q1[c] = a1[c]; q2[c] = a2[c]; q3[c] = a3[c]; }
      *reinterpret_cast<uint4v*>(ws + sw_dst) = q1;
      *reinterpret_cast<uint4v*>(ws + W_PLANE + sw_dst) = q2;
      *reinterpret_cast<uint4v*>(ws + 2 * W_PLANE + sw_dst) = q3;
    };
    auto products = [&](const float* asf, const float* wsf) __attribute__((always_inline)) {
      const char* as = reinterpret_cast<const char*>(asf);
      const char* ws = reinterpret_cast<const char*>(wsf);
      bf16x8 fb[TN][3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          uint4v v;
#pragma unroll
          for (int kp = 0; kp < 4; ++kp)
            v[kp] = *reinterpret_cast<const unsigned*>(ws + p * W_PLANE + ((lh * 4 + kp) * BN + wc + j * 32 + l32) * 4);
          fb[j][p] = __builtin_bit_cast(bf16x8, v);
        }
      bf16x8 fa[TM];
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        if (q == 0 || kPieceA[q] != kPieceA[q - 1]) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
            fa[i] = *reinterpret_cast<const bf16x8*>(as + kPieceA[q] * A_PLANE + (lh * BM + wr + i * 32 + l32) * 16);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j][kPieceB[q]], acc[i][j], 0, 0, 0);
      }
    };
    put(0, As0, Ws0);
    if (KT > 1) fetch(1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int kt = 0; kt < KT; kt += 2) {
      if (kt + 1 < KT) {
        put(kt + 1, As1, Ws1);
        if (kt + 2 < KT) fetch(kt + 2);
      }
      products(As0, Ws0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (kt + 1 < KT) {
        if (kt + 2 < KT) {
          put(kt + 2, As0, Ws0);
          if (kt + 3 < KT) fetch(kt + 3);
        }
        products(As1, Ws1);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    }
  }
  // The loads of a chunk are waited for at the end of the chunk before it; the barrier then
  // also says that every wavefront is done reading the buffer that is refilled next.
  if constexpr (!SPLIT) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  auto kloop = [&]() __attribute__((always_inline)) {
    for (int kt = 0; kt < KT; kt += 2) {
      if (kt + 1 < KT) issue(kt + 1, As1, Ws1);
      compute(As0, Ws0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (kt + 1 < KT) {
        if (kt + 2 < KT) issue(kt + 2, As0, Ws0);
        compute(As1, Ws1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      }
    }
  };
  if constexpr (!SPLIT) kloop();
  // Register r of a block is tile row 8 (r / 4) + 4 (lane / 32) + r % 4 of the block, column
  // lane % 32: Jacobian row p0 + (that row) % PT of the block's position (that row) / PT.
  const int64_t pstride = R * N;  // floats between consecutive Jacobian rows
  const bool full_tile = (p0 + PT <= P) && (col0 + BN <= N) && (r0 + RT <= R);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t pos = r0 + (wrow * TM + i) * PB;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int gc = col0 + wc + j * 32 + l32;
      const float (&d1)[PB] = dr[i][j];
      float* out = a.y_jac + ((int64_t)(p0 + 4 * lh) * R + pos) * N + gc;
      float ss[PB];
#pragma unroll
      for (int b = 0; b < PB; ++b) ss[b] = 0.0f;
      const float* resp = nullptr;
      if constexpr (PARTS) resp = a.res_jac ? a.res_jac + ((int64_t)(p0 + 4 * lh) * R + pos) * N + gc : nullptr;
      auto rows = [&](auto full, auto has_res) __attribute__((always_inline)) {
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
            const bool live = FULL || (p0 + 4 * lh + pl < P && gc < N && pos + b < R);
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
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int pl = 8 * (g % GB) + rr;
            float v = acc[i][j][4 * g + rr];
            const int64_t off = (int64_t)pl * pstride + (int64_t)b * N;
            float* o = out + off;
            if constexpr (FULL) {
              ss[b] = fmaf(v, v, ss[b]);
              float w = d1[b] * v;
              if constexpr (RES) w += rbuf[g & 1][rr];
              __builtin_nontemporal_store(w, o);
            } else if (p0 + 4 * lh + pl < P && pos + b < R) {
              ss[b] = fmaf(v, v, ss[b]);
              if (gc < N) *o = d1[b] * v + (RES ? rbuf[g & 1][rr] : 0.0f);
            }
          }
        }
      };
      if (PARTS && resp != nullptr) {
        if (full_tile) rows(std::true_type{}, std::true_type{});
        else rows(std::false_type{}, std::true_type{});
      } else {
        if (full_tile) rows(std::true_type{}, std::false_type{});
        else rows(std::false_type{}, std::false_type{});
      }
      const int64_t so = ((int64_t)pg * R + pos) * N + gc;
#pragma unroll
      for (int b = 0; b < PB; ++b) {
        const float t = ss[b] + __shfl_xor(ss[b], 32, FOLX_WAVE);
        if (lh == 0 && gc < N && pos + b < R) a.ss[so + (int64_t)b * N] = t;
      }
    }
  }
}

// Finishes the x and lap rows.  On entry y holds z and y_lap the part of zl that is linear in
// the input's lap row (what launch 2 left there).  One float4 per thread.
__global__ __launch_bounds__(256) void dense_wide_finish(float* __restrict__ y, float* __restrict__ y_lap,
                                                         const float* __restrict__ ss, int64_t S4, int32_t PG,
                                                         int32_t act, float prm,
                                                         const float* __restrict__ res,
                                                         const float* __restrict__ res_lap) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= S4) return;
  const float4 z = reinterpret_cast<const float4*>(y)[i];
  float4 zl = reinterpret_cast<const float4*>(y_lap)[i];
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
  if (res_lap) {
    const float4 r = reinterpret_cast<const float4*>(res_lap)[i];
    zl.x += r.x; zl.y += r.y; zl.z += r.z; zl.w += r.w;
  }
  reinterpret_cast<float4*>(y_lap)[i] = zl;
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
  int64_t row_tiles, pos_tiles, blocks, ws_bytes;
  int32_t PG, PT, col_tiles;
};

// What the forms of a dense + activation layer cost: times in us of a 64 x 64 tile and contracted feature on one CU (140
// TFLOP/s over the chip; 233 of fp32 products from bf16 pieces), the work around the K loop in features of that cost, the
// launches, and a MB of a streaming pass.  Fitted to 183 layers per mode (R = 500 .. 40 000, P = 3 .. 183, K = 16 .. 512,
// N = 132 .. 512, all four forms timed): 6 and 7 % rms.
struct WideRates {
  double feature, plain, group8, group16, group32, plain_launches, fused_launches, mb;
};
constexpr WideRates RATES[2] = {{0.015, 46, 50, 36, 29, 9, 13, 0.14}, {0.009, 51, 103, 74, 55, 8, 9, 0.19}};

double wide_time(bool split, int64_t R, int32_t P, int32_t K, int32_t N, int PT) {
  const WideRates& c = RATES[split];
  const int64_t groups = (P + PT - 1) / PT, tiles = (R + BM / PT - 1) / (BM / PT) * groups * ((N + BN - 1) / BN);
  const int64_t rows[3] = {R, 0, R};
  bool small;
  const double around = PT == 8 ? c.group8 : (PT == 16 ? c.group16 : c.group32);
  return c.fused_launches + folx_dense_units(rows, N, split, small) * c.feature * (K + c.plain) +
         8.0 * (double)((tiles + 255) / 256) * c.feature * (K + around) + c.mb * 4e-6 * (double)R * N * (double)(groups + 4);
}

double plain_time(bool split, int64_t R, int32_t P, int32_t K, int32_t N) {
  const WideRates& c = RATES[split];
  const int64_t rows[3] = {R, P * R, R};
  bool small;
  return c.plain_launches + folx_dense_units(rows, N, split, small) * c.feature * (K + c.plain) +
         c.mb * 4e-6 * (double)R * N * 2.0 * (P + 2);
}

// A form replaces the one that needs no estimate (groups of 16 where they divide the positions and leave fewer empty rows than
// 32; the plain product where those leave more than an eighth of the rows empty) only for this much less time: the
// estimate's own error.
constexpr double GAIN = 0.95;

int base_group(int64_t R, int32_t P) { return R % 8 == 0 && (P + 15) / 16 * 16 < (P + 31) / 32 * 32 ? 16 : 32; }

// Jacobian rows of a group for the activation alone.  One group of 8 (P <= 8) would be a layer of short launches, where the
// plain product was as fast.  Of the 183 layers none is more than 5 % slower than in the form that needs no estimate; the
// fewest empty rows alone were 6 to 52 % slower on 30 of them (R = 1788, P = 21, K = 64, N = 300: plain 45 us, groups
// of 8 65; R = 6000, P = 117, K = 64, N = 256: groups of 32 297 us, of 8 329; bf16x3, R = 1968, P = 87, K = 16, N = 256: 50 and 71).
// 180 other layers (R = 250 .. 60 000, P = 2 .. 120): 0.88 of the time of the forms without an estimate in the mean, 0.90 with bf16x3
// (the fewest empty rows: 0.92 and 0.94, more than 3 % slower on 33); four 4 to 6 % slower, among them calls of the same
// form, so within the noise of 20 us.
int act_group(bool split, int64_t R, int32_t P, int32_t K, int32_t N) {
  const int base = base_group(R, P);
  int best = base;
  double least = GAIN * wide_time(split, R, P, K, N, base);
  for (int g = 32; g >= (P > 8 ? 8 : 16); g /= 2) {
    const double t = wide_time(split, R, P, K, N, g);
    if (t < least) { best = g; least = t; }
  }
  return best;
}

bool plan_wide(int64_t R, int32_t P, int32_t K, int32_t N, WidePlan& pl) {
  if (R <= 0 || R % 4 != 0 || P < 1 || K < BK || K % BK != 0 || N <= 128 || N % 4 != 0) return false;
  pl.PT = 32;
  int32_t slabs = 0;
  for (bool split : {false, true}) {  // the workspace serves both product modes: the query and the launch may meet different ones
    const int g = act_group(split, R, P, K, N);
    slabs = std::max(slabs, (P + g - 1) / g);
    if (split == (folx_gemm_mode() == FOLX_HIP_GEMM_BF16X3)) pl.PT = g;
  }
  pl.col_tiles = (N + BN - 1) / BN;
  pl.PG = (P + pl.PT - 1) / pl.PT;
  pl.pos_tiles = (R + BM / pl.PT - 1) / (BM / pl.PT);
  pl.row_tiles = pl.pos_tiles * pl.PG;
  pl.blocks = (pl.row_tiles + NXCD - 1) / NXCD * NXCD * pl.col_tiles;
  if (pl.blocks > 0x7fffffffLL) return false;
  if (R * (int64_t)N / 4 / 256 + 1 > 0x7fffffffLL) return false;
  const int64_t slab = (int64_t)std::max(pl.PG, slabs) * R * N;
  pl.ws_bytes = (slab + 3) / 4 * 4 * 4;
  return true;
}

template <int PT, bool PARTS = false>
int launch_wide(hipStream_t st, const WideParams& a, const WidePlan& pl, float* y, float* y_lap,
                const float* res = nullptr, const float* res_lap = nullptr) {
  const bool split = folx_gemm_mode() == FOLX_HIP_GEMM_BF16X3;
  if (split) dense_wide_kernel<PT, PARTS, true><<<dim3((unsigned)pl.blocks), dim3(NT), 0, st>>>(a);
  if (!split) dense_wide_kernel<PT, PARTS, false><<<dim3((unsigned)pl.blocks), dim3(NT), 0, st>>>(a);
  int rc = folx_launch_status();
  if (rc != FOLX_HIP_OK) return rc;
  const int64_t S4 = a.R * (int64_t)a.N / 4;
  dense_wide_finish<<<dim3((unsigned)((S4 + 255) / 256)), dim3(256), 0, st>>>(
      y, y_lap, a.ss, S4, pl.PG, a.act, a.prm, res, res_lap);
  return folx_launch_status();
}

int run_wide(hipStream_t st, int32_t act, float param, const float* x, const float* jac, const float* lap, const float* W,
             const float* bias, float* y, float* y_jac, float* y_lap, int64_t R, int32_t P, int32_t K, int32_t N, void* workspace,
             int64_t workspace_bytes, const WideParts* parts = nullptr, const float* res = nullptr,
             const float* res_jac = nullptr, const float* res_lap = nullptr, const float* pre = nullptr,
             const float* pre_jac = nullptr, const float* pre_lap = nullptr, int64_t pre_group = 1) {
  WidePlan pl;
  if (act < 0 || !act_fused(act) || !plan_wide(R, P, K, N, pl)) return FOLX_HIP_ENOTSUP;
  if (!x || (!jac && !parts) || !lap || !W || !y || !y_jac || !y_lap) return FOLX_HIP_EINVAL;
  if (!folx_aligned16(jac) || !folx_aligned16(W) || !folx_aligned16(y) || !folx_aligned16(y_lap))
    return FOLX_HIP_ENOTSUP;
  if (!workspace || workspace_bytes < pl.ws_bytes || !folx_aligned16(workspace)) return FOLX_HIP_EINVAL;
  WideParams a;
  a.jac = jac; a.W = W; a.z = y; a.y_jac = y_jac; a.res_jac = res_jac;
  a.pre_jac = pre_jac; a.pre_group = pre_group;
  a.ss = (float*)workspace;
  a.R = R; a.row_tiles = pl.row_tiles; a.pos_tiles = pl.pos_tiles;
  a.P = P; a.K = K; a.N = N; a.col_tiles = pl.col_tiles; a.act = act; a.prm = param;
  // z and the linear part of zl through the plain dense kernel: no Jacobian rows, no residual
  int rc = folx_hip_dense_fwdlap(st, x, nullptr, lap, W, bias, nullptr, nullptr, nullptr, y, nullptr, y_lap, R,
                                 0, K, N);
  if (rc != FOLX_HIP_OK) return rc;
  if (pre) {
    const int64_t S4 = R * (int64_t)N / 4;
    wide_add_pre_kernel<<<dim3((unsigned)((S4 + 255) / 256)), dim3(256), 0, st>>>(y, y_lap, pre, pre_lap, S4, N / 4,
                                                                              pre_group);
    rc = folx_launch_status();
    if (rc != FOLX_HIP_OK) return rc;
  }
  if (parts) {
    a.parts = *parts;
    return pl.PT == 8    ? launch_wide<8, true>(st, a, pl, y, y_lap, res, res_lap)
           : pl.PT == 16 ? launch_wide<16, true>(st, a, pl, y, y_lap, res, res_lap)
                         : launch_wide<32, true>(st, a, pl, y, y_lap, res, res_lap);
  }
  return pl.PT == 8    ? launch_wide<8>(st, a, pl, y, y_lap)
         : pl.PT == 16 ? launch_wide<16>(st, a, pl, y, y_lap)
                       : launch_wide<32>(st, a, pl, y, y_lap);
}

}  // namespace

int folx_dense_act_wide_group(int64_t R, int32_t P, int32_t K, int32_t N) {
  WidePlan pl;
  return plan_wide(R, P, K, N, pl) ? pl.PT : FOLX_HIP_ENOTSUP;
}

int folx_dense_act_wide_faster(int64_t R, int32_t P, int32_t K, int32_t N, int32_t plain) {
  WidePlan pl;
  if (!plan_wide(R, P, K, N, pl)) return FOLX_HIP_ENOTSUP;
  const int base = base_group(R, P);
  if ((P + base - 1) / base * base <= 1.125 * P) return 1;
  const bool split = folx_gemm_mode() == FOLX_HIP_GEMM_BF16X3;
  return wide_time(split, R, P, K, N, pl.PT) < GAIN * plain_time(split, R, P, plain, N);
}

int64_t folx_dense_act_wide_ws_bytes(int64_t R, int32_t P, int32_t K, int32_t N) {
  WidePlan pl;
  if (!plan_wide(R, P, K, N, pl)) return FOLX_HIP_ENOTSUP;
  return pl.ws_bytes;
}

int folx_dense_act_wide(hipStream_t st, int32_t act, float param, const float* x, const float* jac, const float* lap,
                        const float* W, const float* bias, float* y, float* y_jac, float* y_lap, int64_t R,
                        int32_t P, int32_t K, int32_t N, void* workspace, int64_t workspace_bytes) {
  if (act < 0) return FOLX_HIP_ENOTSUP;
  const int64_t need = folx_wide_pieces_ws_bytes(R, P, K, N);
  if (need > 0 && workspace_bytes >= need)
    return folx_wide_pieces(st, act, param, x, jac, lap, nullptr, W, bias, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 1, y,
                            y_jac, y_lap, R, P, K, N, workspace, workspace_bytes);
  return run_wide(st, act, param, x, jac, lap, W, bias, y, y_jac, y_lap, R, P, K, N,
                  workspace, workspace_bytes);
}

extern "C" int folx_hip_dense_act_parts_fwdlap(void* stream, int32_t act, float param, const float* x,
                                               const float* lap, int32_t n_parts, const float* const* jac_parts,
                                               const int32_t* widths, const int32_t* broadcast, int32_t group,
                                               const float* W, const float* bias, const float* res,
                                               const float* res_jac, const float* res_lap, const float* pre,
                                               const float* pre_jac, const float* pre_lap, float* y,
                                               float* y_jac, float* y_lap, int64_t R, int32_t P, int32_t N,
                                               void* workspace, int64_t workspace_bytes) {
  if (R < 0 || P < 0 || N <= 0 || n_parts < 1 || group < 1 || !jac_parts || !widths || !broadcast)
    return FOLX_HIP_EINVAL;
  if ((res != nullptr) != (res_jac != nullptr) || (res != nullptr) != (res_lap != nullptr)) return FOLX_HIP_EINVAL;
  if ((pre != nullptr) != (pre_jac != nullptr) || (pre != nullptr) != (pre_lap != nullptr)) return FOLX_HIP_EINVAL;
  if (!folx_aligned16(res) || !folx_aligned16(res_lap) || !folx_aligned16(pre) || !folx_aligned16(pre_lap))
    return FOLX_HIP_ENOTSUP;
  if (n_parts > MAX_PARTS || act < 0 || R % group != 0) return FOLX_HIP_ENOTSUP;
  WideParts parts;
  parts.n = n_parts;
  parts.group = group;
  int32_t K = 0;
  for (int i = 0; i < n_parts; ++i) {
    if (widths[i] <= 0 || widths[i] % BK != 0) return FOLX_HIP_ENOTSUP;
    if (!jac_parts[i]) return FOLX_HIP_EINVAL;
    if (!folx_aligned16(jac_parts[i])) return FOLX_HIP_ENOTSUP;
    parts.jac[i] = jac_parts[i];
    parts.width[i] = widths[i];
    parts.bcast[i] = broadcast[i] ? 1 : 0;
    parts.pstride[i] = (broadcast[i] ? R / group : R) * (int64_t)widths[i];
    K += widths[i];
    parts.kend[i] = K;
  }
  for (int i = n_parts; i < MAX_PARTS; ++i) {
    parts.jac[i] = nullptr; parts.width[i] = 0; parts.bcast[i] = 0; parts.pstride[i] = 0; parts.kend[i] = K;
  }
  const int64_t need = folx_wide_pieces_ws_bytes(R, P, K, N);
  if (need > 0 && workspace_bytes >= need)
    return folx_wide_pieces((hipStream_t)stream, act, param, x, nullptr, lap, &parts, W, bias, res, res_jac, res_lap, pre, pre_jac,
                            pre_lap, group, y, y_jac, y_lap, R, P, K, N, workspace, workspace_bytes);
  return run_wide((hipStream_t)stream, act, param, x, nullptr, lap, W, bias, y, y_jac,
                  y_lap, R, P, K, N, workspace, workspace_bytes, &parts, res, res_jac, res_lap, pre, pre_jac, pre_lap,
                  group);
}

