// Multi-head self attention with Laplacian:  o = softmax(q k^T) v  and its Jacobian rows
// and Laplacian, one workgroup per (walker, head): mhsa_small_kernel for n <= 16 (its mapping stands there), mhsa_kernel beyond.
//
// Algebra per Jacobian row c (the factored form of the rule):
//   s'_c = q'_c k^T + q k'_c^T          p'_c = p * (s'_c - rowsum(p * s'_c))
//   o'_c = p v'_c + p'_c v
//   lap_o = p lap_v + pL v                                   (pL: same as p'_c with lap_q, lap_k)
//         + [ X + p * (2 G - u - rowsum(p * 2 G)) ] v + 2 sum_c p'_c v'_c
//   X = sum_c p'_c * (s'_c - rowsum(p s'_c)),  G = sum_c q'_c k'_c^T,  u = sum_c rowsum(p'_c s'_c)
// i.e. six n x n x d matrix products per row, all on v_mfma_f32_16x16x4_f32.  With an edge
// bias e (s = q k^T + e) the rows e'_c and lap_e are added to s'_c and to the Laplacian's
// first-order part; they have no second-order contribution.
//
// Mapping of mhsa_kernel: wavefront w owns query rows [16 w, 16 w + 16) and every key column, so all
// row reductions stay inside 16-lane groups of one wavefront.  k, v and the current
// k'_c, v'_c tiles are shared through LDS (the next pair waits in registers; a single LDS
// copy keeps the workgroup under 40 KB, so four workgroups share a CU); q, q'_c and p live in
// registers in MFMA A-operand layout; p'_c goes through a wavefront-private LDS tile to
// turn the MFMA result layout into the A-operand layout.  As in the GEMM, the k index
// inside a group of 16 is permuted (lane l, register r <-> k = 4 (l / 16) + r) so that A
// operands are fetched with 128-bit reads.
#include "common.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Sum and maximum over the 16 lanes of a row, by DPP: quad permutes (lane ^ 1, lane ^ 2), then the two mirrors, which
// meet equal values in every quad (half of 8) by then.  Vector instructions only, where a shuffle is a trip through LDS:
// mhsa_kernel on 1200 pairs of 17 x 64, P = 51: 797 -> 766 us, on 1024 of 32 x 64, P = 96: 745 -> 725 us.
template <int CTRL>
__device__ __forceinline__ float dpp16(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum16(float v) {
  v += dpp16<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp16<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp16<0x141>(v);  // row_half_mirror
  v += dpp16<0x140>(v);  // row_mirror
  return v;
}
__device__ __forceinline__ float max16(float v) {
  v = fmaxf(v, dpp16<0xB1>(v));
  v = fmaxf(v, dpp16<0x4E>(v));
  v = fmaxf(v, dpp16<0x141>(v));
  v = fmaxf(v, dpp16<0x140>(v));
  return v;
}
__device__ __forceinline__ float f4get(const float4& v, int r) {
  return r == 0 ? v.x : (r == 1 ? v.y : (r == 2 ? v.z : v.w));
}

struct MhsaArgs {
  const float *q, *qj, *ql, *k, *kj, *kl, *v, *vj, *vl;
  const float *e, *ej, *el;  // optional edge bias [B][n][H][n] and its Jacobian rows / Laplacian
  const uint8_t *mask, *imask;
  float *o, *oj, *ol;
  int64_t B;
  int32_t n, H, d, P;
};

// FAST: n = 16 NW, d = 16 DT and no masks -- every bounds / mask test folds away.
template <int NW, int DT, bool EDGE, bool FAST>
__global__ __launch_bounds__(FOLX_WAVE * NW) void mhsa_kernel(MhsaArgs a) {
  constexpr int NP = 16 * NW;   // padded sequence length
  constexpr int DP = 16 * DT;   // padded head dim
  constexpr int DS = DP + 4;    // LDS row stride of (n x d) tiles
  constexpr int NS = NP + 4;    // LDS row stride of the per-wavefront (16 x n) tiles
  constexpr int NT = FOLX_WAVE * NW;
  constexpr int TILE4 = NP * DP / 4;                 // float4 per (n x d) tile
  constexpr int LD4 = (TILE4 + NT - 1) / NT;         // float4 per thread per tile
  constexpr float BIG = 1e20f;

  __shared__ __attribute__((aligned(16))) float ks[NP * DS];
  __shared__ __attribute__((aligned(16))) float vs[NP * DS];
  __shared__ __attribute__((aligned(16))) float kjs1[NP * DS];
  __shared__ __attribute__((aligned(16))) float vjs1[NP * DS];
  __shared__ __attribute__((aligned(16))) float pst[NW][16 * NS];

  const int tid = threadIdx.x;
  const int lane = tid % FOLX_WAVE;
  const int w = tid / FOLX_WAVE;
  const int l16 = lane % 16;
  const int lg = lane / 16;
  const int64_t b = blockIdx.x / a.H;
  const int h = blockIdx.x % a.H;
  const int n = a.n, d = a.d, H = a.H, P = a.P;
  const int64_t B = a.B;
  const int64_t tok = (int64_t)H * d;                 // stride between electrons
  const int64_t base = (b * n) * tok + (int64_t)h * d;  // offset of (b, 0, h, 0)
  const int64_t slice = B * n * tok;                  // stride between Jacobian rows

  auto valid = [&](int i) -> bool {
    if constexpr (FAST) return true;
    return i < n && (a.mask == nullptr || a.mask[b * n + i] != 0);
  };
  // edge-bias entries of this lane in result layout: row 16 w + 4 lg + r, column 16 jt + l16
  const int64_t etok = (int64_t)H * n;
  const int64_t ebase = (b * n) * etok + (int64_t)h * n;
  const int64_t eslice = B * n * etok;
  auto edge_add = [&](const float* src, floatx4* acc) {
#pragma unroll
    for (int jt = 0; jt < NW; ++jt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * w + 4 * lg + r, col = 16 * jt + l16;
        if (FAST || (row < n && col < n)) acc[jt][r] += src[ebase + (int64_t)row * etok + col];
      }
  };

  // cooperative load of an (n x d) tile into LDS, rows of padding electrons zeroed
  float4 rk[LD4], rv[LD4];
  auto tile_load = [&](const float* src, float4* reg, bool mask_rows) {
#pragma unroll
    for (int i = 0; i < LD4; ++i) {
      const int idx = tid + NT * i;
      const int j = idx / (DP / 4);
      const int a4 = (idx % (DP / 4)) * 4;
      float4 val = make_float4(0.f, 0.f, 0.f, 0.f);
      if (FAST || (idx < TILE4 && j < n && a4 < d && (!mask_rows || valid(j))))
        val = folx_ld_stream4(src + base + (int64_t)j * tok + a4);  // every tile is read once
      reg[i] = val;
    }
  };
  auto tile_store = [&](float* dst, const float4* reg) {
#pragma unroll
    for (int i = 0; i < LD4; ++i) {
      const int idx = tid + NT * i;
      const int j = idx / (DP / 4);
      const int a4 = (idx % (DP / 4)) * 4;
      if (FAST || idx < TILE4) *reinterpret_cast<float4*>(dst + j * DS + a4) = reg[i];
    }
  };
  // A-operand registers of this wavefront's 16 rows of an (n x d) array:
  // reg[t] = src[row][4 lg + 16 t .. + 3]
  const int qrow = 16 * w + l16;
  auto rows_load = [&](const float* src, float4* reg, bool mask_rows) {
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int a4 = 4 * lg + 16 * t;
      float4 val = make_float4(0.f, 0.f, 0.f, 0.f);
      if (FAST || (qrow < n && a4 < d && (!mask_rows || valid(qrow))))
        val = folx_ld_stream4(src + base + (int64_t)qrow * tok + a4);
      reg[t] = val;
    }
  };

  // ---- forward ---------------------------------------------------------------------------
  tile_load(a.k, rk, false);
  tile_load(a.v, rv, false);
  tile_store(ks, rk);
  tile_store(vs, rv);
  float4 qa[DT];
  rows_load(a.q, qa, false);
  __syncthreads();

  bool rvalid[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) rvalid[r] = valid(16 * w + 4 * lg + r);
  bool cvalid[NW], cexist[NW];
#pragma unroll
  for (int jt = 0; jt < NW; ++jt) { cexist[jt] = FAST || (16 * jt + l16) < n; cvalid[jt] = valid(16 * jt + l16); }

  // s = q k^T  (A = q registers, B = k from LDS)
  auto qk_product = [&](const float4* areg, const float* btile, floatx4* acc) {
#pragma unroll
    for (int jt = 0; jt < NW; ++jt) {
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const float4 bv = *reinterpret_cast<const float4*>(&btile[(16 * jt + l16) * DS + 4 * lg + 16 * t]);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(f4get(areg[t], r), f4get(bv, r), acc[jt], 0, 0, 0);
      }
    }
  };
  // o = p v  (A = p-like registers [NW float4], B = v-like tile from LDS)
  auto pv_product = [&](const float4* areg, const float* btile, floatx4* acc) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int t = 0; t < NW; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float bv = btile[(4 * lg + 16 * t + r) * DS + 16 * dt + l16];
          acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(f4get(areg[t], r), bv, acc[dt], 0, 0, 0);
        }
      }
    }
  };
  // result layout (row 4 lg + r, column 16 jt + l16) -> A-operand layout through LDS
  auto to_a_layout = [&](const floatx4* c, float4* areg) {
    float* st = pst[w];
#pragma unroll
    for (int jt = 0; jt < NW; ++jt)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[(4 * lg + r) * NS + 16 * jt + l16] = c[jt][r];
    // The tile is private to this wavefront, whose LDS accesses complete in issue order:
    // a wavefront-scope fence (no reordering by the compiler) is all the exchange needs.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int t = 0; t < NW; ++t) areg[t] = *reinterpret_cast<const float4*>(&st[l16 * NS + 4 * lg + 16 * t]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  floatx4 pc[NW];  // softmax probabilities, result layout
  {
    floatx4 s[NW];
#pragma unroll
    for (int jt = 0; jt < NW; ++jt) s[jt] = floatx4{0.f, 0.f, 0.f, 0.f};
    qk_product(qa, ks, s);
    if constexpr (EDGE) edge_add(a.e, s);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float mx = -INFINITY;
#pragma unroll
      for (int jt = 0; jt < NW; ++jt) {
        float sv = s[jt][r];
        if (!cexist[jt]) sv = -INFINITY;
        else if (!(rvalid[r] && cvalid[jt])) sv = -BIG;
        s[jt][r] = sv;
        mx = fmaxf(mx, sv);
      }
      mx = max16(mx);
      float sum = 0.0f;
#pragma unroll
      for (int jt = 0; jt < NW; ++jt) {
        const float e = cexist[jt] ? expf(s[jt][r] - mx) : 0.0f;
        s[jt][r] = e;
        sum += e;
      }
      sum = sum16(sum);
      const float inv = 1.0f / sum;
#pragma unroll
      for (int jt = 0; jt < NW; ++jt) pc[jt][r] = s[jt][r] * inv;
    }
  }
  float4 pa[NW];
  to_a_layout(pc, pa);

  floatx4 oc[DT];  // o, result layout: row 4 lg + r, column 16 dt + l16
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  pv_product(pa, vs, oc);
  // per-lane offset of (row 16 w + 4 lg, column l16) inside one (n, H, d) slice
  const int64_t out_off = base + (int64_t)(16 * w + 4 * lg) * tok + l16;
  auto out_store = [&](float* dst, const floatx4* c) {
    if constexpr (FAST) {
      float* p = dst + out_off;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) __builtin_nontemporal_store(c[dt][r], &p[16 * dt]);
        p += tok;
      }
    } else {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * w + 4 * lg + r, col = 16 * dt + l16;
          if (row < n && col < d) dst[base + (int64_t)row * tok + col] = c[dt][r];
        }
    }
  };
  out_store(a.o, oc);

  // ---- Jacobian rows and Laplacian -------------------------------------------------------
  floatx4 G[NW], X[NW], O2[DT], OL[DT];
  float u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int jt = 0; jt < NW; ++jt) { G[jt] = floatx4{0.f, 0.f, 0.f, 0.f}; X[jt] = G[jt]; }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) { O2[dt] = floatx4{0.f, 0.f, 0.f, 0.f}; OL[dt] = O2[dt]; }

  // pass c < P: Jacobian row c; pass c == P: the Laplacians take the place of the row
  auto active = [&](int c) -> bool {
    if constexpr (FAST) return true;
    return c == P || a.imask == nullptr || a.imask[(int64_t)c * B + b] != 0;
  };
  auto src_of = [&](const float* jac, const float* lap, int c) -> const float* {
    return c == P ? lap : jac + (int64_t)c * slice;
  };

  float4 qja[DT];
  if (active(0)) {
    tile_load(src_of(a.kj, a.kl, 0), rk, true);
    tile_load(src_of(a.vj, a.vl, 0), rv, true);
    rows_load(src_of(a.qj, a.ql, 0), qja, true);
    tile_store(kjs1, rk);
    tile_store(vjs1, rv);
  }
  __syncthreads();

  for (int c = 0; c <= P; ++c) {
    const bool act = active(c);
    const bool nact = c < P && active(c + 1);
    float4 qjn[DT];
    if (nact) {
      tile_load(src_of(a.kj, a.kl, c + 1), rk, true);
      tile_load(src_of(a.vj, a.vl, c + 1), rv, true);
      rows_load(src_of(a.qj, a.ql, c + 1), qjn, true);
    }
    if (act) {
      const bool is_lap = c == P;
      // s'_c = q'_c k^T + q k'_c^T ;  G += q'_c k'_c^T
      floatx4 sj[NW];
#pragma unroll
      for (int jt = 0; jt < NW; ++jt) sj[jt] = floatx4{0.f, 0.f, 0.f, 0.f};
      qk_product(qja, ks, sj);
      qk_product(qa, kjs1, sj);
      if constexpr (EDGE) edge_add(is_lap ? a.el : a.ej + (int64_t)c * eslice, sj);
      if (!is_lap) qk_product(qja, kjs1, G);
      // p'_c = p * (s'_c - rowsum(p s'_c))
      floatx4 pj[NW];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float rs = 0.0f;
#pragma unroll
        for (int jt = 0; jt < NW; ++jt) rs += pc[jt][r] * sj[jt][r];
        rs = sum16(rs);
        float us = 0.0f;
#pragma unroll
        for (int jt = 0; jt < NW; ++jt) {
          const float dlt = sj[jt][r] - rs;
          const float pv = pc[jt][r] * dlt;
          pj[jt][r] = pv;
          if (!is_lap) { X[jt][r] += pv * dlt; us += pv * sj[jt][r]; }
        }
        u[r] += us;  // lane-partial; reduced over the 16-lane group at the end
      }
      float4 pja[NW];
      to_a_layout(pj, pja);
      // o'_c = p v'_c + p'_c v ;  O2 += p'_c v'_c
      floatx4 ojc[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) ojc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
      pv_product(pa, vjs1, ojc);
      pv_product(pja, vs, ojc);
      if (!is_lap) {
        pv_product(pja, vjs1, O2);
        out_store(a.oj + (int64_t)c * slice, ojc);
      } else {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) OL[dt] = ojc[dt];
      }
    } else {
      // inactive coordinate: its Jacobian row is zero and it adds nothing to the Laplacian
      floatx4 z[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) z[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
      out_store(a.oj + (int64_t)c * slice, z);
    }
    __syncthreads();  // every wavefront is done with the current k', v' tiles
    if (nact) {
      tile_store(kjs1, rk);
      tile_store(vjs1, rv);
#pragma unroll
      for (int t = 0; t < DT; ++t) qja[t] = qjn[t];
    }
    __syncthreads();
  }

  // ---- second-order part:  [X + p * (2 G - u - rowsum(2 p G))] v + 2 O2 ------------------
  floatx4 pi[NW];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float ur = sum16(u[r]);
    float rs = 0.0f;
#pragma unroll
    for (int jt = 0; jt < NW; ++jt) rs += pc[jt][r] * 2.0f * G[jt][r];
    rs = sum16(rs);
#pragma unroll
    for (int jt = 0; jt < NW; ++jt) pi[jt][r] = X[jt][r] + pc[jt][r] * (2.0f * G[jt][r] - ur - rs);
  }
  float4 pia[NW];
  to_a_layout(pi, pia);
  pv_product(pia, vs, OL);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) OL[dt][r] += 2.0f * O2[dt][r];
  out_store(a.ol, OL);
}

// n <= 16: one wavefront covers all query rows of a (walker, head) pair, so its rows c need nothing from its neighbours:
// q'_c, k'_c and v'_c go from memory straight into MFMA operand registers and the W wavefronts of a workgroup take the rows
// c = w, w + W, ... with every sum over rows in registers, added through LDS once at the end (k and v wait in LDS, the same
// for all of them: 168 registers, twelve wavefronts on a CU; with a bias or masks and four blocks of features 182 to 194,
// eight wavefronts).  Rows and columns of the padding are lanes whose buffer offset
// lies past the descriptor's end: they read zeros and their stores are dropped, so no access is tested.  DT = 1, 2 or 4
// blocks of 16 features.
// Bound by HBM (16 n d bytes per pair and row, at 4.6-5.3 TB/s), for few pairs by the latency of a wavefront's rows.  One
// wavefront per pair with the tiles of mhsa_kernel (two barriers and an LDS copy of k', v' per row) was bound by that chain:
// 1200 pairs of 13 x 64, P = 39: 300 -> 139 us; 256 of 10 x 64, P = 30: 112 -> 24 us; 2048 of 16 x 16, P = 48: 146 -> 94 us;
// 16000 of 16 x 64, P = 48: 2.69 -> 2.56 ms; 33 to 48 features run as four blocks: 1200 of 13 x 48, P = 39: 232 -> 108 us.  With a bias, masks, both (former kernel -> this; in parentheses held to 168
// registers, 15 to 32 of them spilled, and the bias loaded where it is added): 1200 pairs of 13 x 64, P = 39: 414 -> 150 us
// (202), 742 -> 153 (210), 847 -> 158 (286); 2048 of 12 x 36, P = 36: 202 -> 162 (275), 503 -> 189 (280), 368 -> 192 (392);
// 4096 of 16 x 64, P = 48: 752 -> 690 (844), 2053 -> 617 (832), 2324 -> 685 (1163).
constexpr int NXCD = 8;
constexpr uint32_t FAR = 0x40000000u;  // past every descriptor's end, also with the row and piece offsets added
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

template <int DT, bool EDGE, bool MASKED>
__global__ __launch_bounds__(512, DT == 4 && (EDGE || MASKED) ? 2 : 3) void mhsa_small_kernel(MhsaArgs a) {
  constexpr float BIG = 1e20f;
  constexpr int NS = 20;           // LDS row stride of a 16 x 16 tile
  constexpr int NRED = 12 + 4 * DT;
  const int W = blockDim.x / FOLX_WAVE;
  constexpr int KS = 16 * DT + 4;  // row stride of the copies of k and v (the same for every wavefront; read once per row)
  extern __shared__ __attribute__((aligned(16))) float lds[];  // [W][16 NS] tiles, later [W - 1][NRED][64] sums
  __shared__ __attribute__((aligned(16))) float ksh[16 * KS];
  __shared__ __attribute__((aligned(16))) float vsh[16 * KS];

  const int lane = threadIdx.x % FOLX_WAVE;
  const int w = folx_wave_id();
  const int l16 = lane % 16;
  const int lg = lane / 16;
  // ids are dealt round-robin to the XCDs: consecutive pairs (the heads of a walker share cache lines when d < 32) go to one
  const int64_t pairs = a.B * a.H, per = (pairs + NXCD - 1) / NXCD;
  const int64_t pair = (int64_t)(blockIdx.x % NXCD) * per + blockIdx.x / NXCD;
  if (pair >= pairs) return;
  const int64_t b = pair / a.H;
  const int h = (int)(pair % a.H);
  const int n = a.n, d = a.d, H = a.H, P = a.P;
  const int64_t B = a.B;
  const int32_t tok = H * d;
  const int64_t base = (b * n) * tok + (int64_t)h * d;
  const int64_t slice = B * n * tok;
  const uint32_t bytes = (uint32_t)(((int64_t)n * tok - (int64_t)h * d) * 4);  // from (b, 0, h, 0) to the walker's end

  auto rsrc = [&](const float* p) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p) + base, 0, bytes, 0x00027000);
  };
  auto valid = [&](int i) __attribute__((always_inline)) -> bool {
    return i < n && (!MASKED || a.mask == nullptr || a.mask[b * n + i] != 0);
  };
  // byte offsets of this lane: row l16, piece 4 lg of 16 t (A / k layout); rows 4 lg + r, columns DT l16 .. + DT - 1 (v and
  // result: column l16 of block dt stands for DT l16 + dt, so that a lane's DT columns are one access)
  uint32_t ao[DT], vo[4], aoj[DT], voj[4];  // ..j: rows of masked inputs read zeros as well
  const bool arow = valid(l16);
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    const bool in = l16 < n && 16 * t + 4 * lg < d;
    ao[t] = in ? (uint32_t)(l16 * tok + 16 * t + 4 * lg) * 4u : FAR;
    aoj[t] = MASKED && !arow ? FAR : ao[t];
  }
  bool rvalid[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 4 * lg + r;
    rvalid[r] = valid(row);
    vo[r] = row < n && DT * l16 < d ? (uint32_t)(row * tok + DT * l16) * 4u : FAR;
    voj[r] = MASKED && !rvalid[r] ? FAR : vo[r];
  }
  auto load_rows = [&](const float* src, const uint32_t (&off)[DT], float4 (&reg)[DT]) __attribute__((always_inline)) {
    const auto rs = rsrc(src);
#pragma unroll
    for (int t = 0; t < DT; ++t)
      reg[t] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, off[t], 0, 0));
  };
  auto load_v = [&](const float* src, const uint32_t (&off)[4], float (&reg)[DT][4]) __attribute__((always_inline)) {
    const auto rs = rsrc(src);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (DT == 4) {
        const uintx4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, off[r], 0, 0);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) reg[dt][r] = __uint_as_float(v[dt]);
      } else if constexpr (DT == 2) {
        const uintx2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, off[r], 0, 0);
        reg[0][r] = __uint_as_float(v[0]);
        reg[1][r] = __uint_as_float(v[1]);
      } else {
        reg[0][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off[r], 0, 0));
      }
    }
  };
  auto store = [&](float* dst, const floatx4 (&c)[DT]) __attribute__((always_inline)) {
    const auto rs = rsrc(dst);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      unsigned x[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const float v = c[dt][r];
        x[dt] = __float_as_uint(v);
      }
      if constexpr (DT == 4) {
        uintx4 v;
        v[0] = x[0]; v[1] = x[1]; v[2] = x[2]; v[3] = x[3];
        __builtin_amdgcn_raw_buffer_store_b128(v, rs, vo[r], 0, 2);
      } else if constexpr (DT == 2) {
        uintx2 v;
        v[0] = x[0]; v[1] = x[1];
        __builtin_amdgcn_raw_buffer_store_b64(v, rs, vo[r], 0, 2);
      } else {
        __builtin_amdgcn_raw_buffer_store_b32(x[0], rs, vo[r], 0, 2);
      }
    }
  };
  const int64_t etok = (int64_t)H * n, ebase = (b * n) * etok + (int64_t)h * n, eslice = B * n * etok;
  const uint32_t ebytes = (uint32_t)(((int64_t)n * etok - (int64_t)h * n) * 4);
  uint32_t eo[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) eo[r] = 4 * lg + r < n && l16 < n ? (uint32_t)((4 * lg + r) * (int32_t)etok + l16) * 4u : FAR;
  auto load_e = [&](const float* src) __attribute__((always_inline)) -> floatx4 {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src) + ebase, 0, ebytes, 0x00027000);
    floatx4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, eo[r], 0, 0));
    return v;
  };
  auto qk = [&](const float4 (&x)[DT], const float4 (&y)[DT], floatx4& acc) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(f4get(x[t], r), f4get(y[t], r), acc, 0, 0, 0);
  };
  auto pv = [&](const float4& p, const float (&y)[DT][4], floatx4 (&acc)[DT]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(f4get(p, r), y[dt][r], acc[dt], 0, 0, 0);
  };
  float* st = lds + w * 16 * NS;
  auto to_a = [&](const floatx4& c) __attribute__((always_inline)) -> float4 {
#pragma unroll
    for (int r = 0; r < 4; ++r) st[(4 * lg + r) * NS + l16] = c[r];
    // private to this wavefront, whose LDS accesses complete in issue order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float4 v = *reinterpret_cast<const float4*>(&st[l16 * NS + 4 * lg]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return v;
  };

  // pass c < P: Jacobian row c; pass c == P: the Laplacians take the place of the row
  auto active = [&](int c) __attribute__((always_inline)) -> bool {
    return !MASKED || c == P || a.imask == nullptr || a.imask[(int64_t)c * B + b] != 0;
  };
  auto src_of = [&](const float* jac, const float* lap, int c) __attribute__((always_inline)) -> const float* {
    return c == P ? lap : jac + (int64_t)c * slice;
  };
  // The next row's q', k' (and bias) are asked for as soon as the products that read this row's are issued, and its v'
  // behind the other three: half a row of matrix work ahead in the same registers, the rest of the latency is other
  // wavefronts' time.  (Loads complete in order: a bias loaded where it is added would wait for the next row's operands.)
  float4 qj[DT], kj[DT];
  floatx4 ej;
  float vj[DT][4];
  auto fetch_qk = [&](int c) __attribute__((always_inline)) {
    load_rows(src_of(a.qj, a.ql, c), aoj, qj);
    load_rows(src_of(a.kj, a.kl, c), aoj, kj);
    if constexpr (EDGE) ej = load_e(c == P ? a.el : a.ej + (int64_t)c * eslice);
  };
  auto fetch_v = [&](int c) __attribute__((always_inline)) { load_v(src_of(a.vj, a.vl, c), voj, vj); };

  float4 qa[DT];
  load_rows(a.q, ao, qa);
  floatx4 e0;
  if constexpr (EDGE) e0 = load_e(a.e);
  if (w == 0) {
    float4 kr[DT];
    float vr[DT][4];
    load_rows(a.k, ao, kr);
    load_v(a.v, vo, vr);
#pragma unroll
    for (int t = 0; t < DT; ++t) *reinterpret_cast<float4*>(&ksh[l16 * KS + 16 * t + 4 * lg]) = kr[t];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) vsh[(4 * lg + r) * KS + DT * l16 + dt] = vr[dt][r];
  }
  auto k_rows = [&](float4 (&kb)[DT]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < DT; ++t) kb[t] = *reinterpret_cast<const float4*>(&ksh[l16 * KS + 16 * t + 4 * lg]);
  };
  auto v_rows = [&](float (&vb)[DT][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* p = &vsh[(4 * lg + r) * KS + DT * l16];
      if constexpr (DT == 4) {
        const float4 x = *reinterpret_cast<const float4*>(p);
        vb[0][r] = x.x; vb[1][r] = x.y; vb[2][r] = x.z; vb[3][r] = x.w;
      } else {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vb[dt][r] = p[dt];
      }
    }
  };
  if (w <= P && active(w)) {
    fetch_qk(w);
    fetch_v(w);
  }

  const bool cexist = l16 < n, cvalid = arow;
  floatx4 pc = floatx4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  {
    float4 kb[DT];
    k_rows(kb);
    qk(qa, kb, pc);
  }
  if constexpr (EDGE) pc += e0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float sv = pc[r];
    if (!cexist) sv = -INFINITY;
    else if (!(rvalid[r] && cvalid)) sv = -BIG;
    const float mx = max16(sv);
    const float e = cexist ? expf(sv - mx) : 0.0f;
    pc[r] = e * (1.0f / sum16(e));
  }
  const float4 pa = to_a(pc);
  if (w == 0) {
    floatx4 oc[DT];
    float vb[DT][4];
    v_rows(vb);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    pv(pa, vb, oc);
    store(a.o, oc);
  }

  floatx4 G = floatx4{0.f, 0.f, 0.f, 0.f}, X = G, O2[DT], OL[DT];
  float u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) { O2[dt] = G; OL[dt] = G; }
  for (int c = w; c <= P; c += W) {
    const bool act = active(c), next = c + W <= P && active(c + W);
    floatx4 oj[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oj[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (act) {
      const bool is_lap = c == P;
      floatx4 sj = floatx4{0.f, 0.f, 0.f, 0.f};
      {
        float4 kb[DT];
        k_rows(kb);
        qk(qj, kb, sj);
      }
      qk(qa, kj, sj);
      if (!is_lap) qk(qj, kj, G);
      if constexpr (EDGE) sj += ej;
      if (next) fetch_qk(c + W);
      floatx4 pj;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float rs = sum16(pc[r] * sj[r]);
        const float dlt = sj[r] - rs;
        pj[r] = pc[r] * dlt;
        if (!is_lap) {
          X[r] += pj[r] * dlt;
          u[r] += pj[r] * sj[r];  // lane-partial; reduced over the 16 lanes at the end
        }
      }
      const float4 pja = to_a(pj);
      {
        float vb[DT][4];
        v_rows(vb);
        pv(pja, vb, oj);
      }
      pv(pa, vj, oj);
      if (!is_lap) {
        pv(pja, vj, O2);
      } else {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) OL[dt] = oj[dt];
      }
    } else if (next) {
      fetch_qk(c + W);
    }
    if (next) fetch_v(c + W);
    if (c < P) store(a.oj + (int64_t)c * slice, oj);  // zeros for an inactive coordinate
  }

  // sums over rows: wavefronts 1 .. W - 1 leave theirs in LDS, wavefront 0 adds them in order
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) O2[dt][r] = 2.0f * O2[dt][r] + OL[dt][r];
  __syncthreads();
  if (w > 0) {
    float* o = lds + (w - 1) * NRED * 64 + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[r * 64] = G[r];
      o[(4 + r) * 64] = X[r];
      o[(8 + r) * 64] = u[r];
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[(12 + 4 * dt + r) * 64] = O2[dt][r];
  }
  __syncthreads();
  if (w > 0) return;
  for (int i = 0; i < W - 1; ++i) {
    const float* o = lds + i * NRED * 64 + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      G[r] += o[r * 64];
      X[r] += o[(4 + r) * 64];
      u[r] += o[(8 + r) * 64];
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) O2[dt][r] += o[(12 + 4 * dt + r) * 64];
  }
  // second-order part:  [X + p * (2 G - u - rowsum(2 p G))] v + (2 O2 + first-order part)
  floatx4 pi;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float ur = sum16(u[r]);
    const float rs = sum16(pc[r] * 2.0f * G[r]);
    pi[r] = X[r] + pc[r] * (2.0f * G[r] - ur - rs);
  }
  // the tile of this wavefront may alias sums that it has read: same wavefront, LDS in order
  const float4 pia = to_a(pi);
  float vb[DT][4];
  v_rows(vb);
  pv(pia, vb, O2);
  store(a.ol, O2);
}

// W wavefronts per pair: twelve fit a CU, three workgroups of four; eight share the rows where a CU gets one pair at most.
// us for W = 1, 4, 8, pairs of 16 x 16: 192, P = 16: 16.6, 8.3, 7.8; P = 48: 41.7, 16.5, 13.0; 512, P = 48: 45.9, 21.8, 20.7.  Of 10 x 64:
// 192, P = 16: 34.8, 15.6, 16.7; P = 48: 96, 32.1, 29.7; 384, P = 48: 98, 49.0, 53.1.  Below eight rows the copies and sums are
// most of what four wavefronts do: 8192 pairs of 10 x 64, P = 7: 154, 172 (W = 4); few pairs would still be faster with four (64, P = 6: 17, 10).
template <int DT>
int launch_mhsa_small(hipStream_t st, const MhsaArgs& a) {
  const int64_t pairs = a.B * a.H;
  if (pairs > 0x7ffffff0LL) return FOLX_HIP_ENOTSUP;
  const int W = a.P < 8 ? 1 : (pairs <= 192 && a.P >= 16 ? 8 : 4);
  const size_t tiles = (size_t)W * 16 * 20, sums = (size_t)(W - 1) * (12 + 4 * DT) * 64;
  const size_t shm = 4 * (tiles > sums ? tiles : sums);
  const dim3 grid((unsigned)((pairs + NXCD - 1) / NXCD * NXCD)), block((unsigned)(FOLX_WAVE * W));
  const bool masked = a.mask != nullptr || a.imask != nullptr;
  if (a.e != nullptr) {
    if (masked) mhsa_small_kernel<DT, true, true><<<grid, block, shm, st>>>(a);
    else mhsa_small_kernel<DT, true, false><<<grid, block, shm, st>>>(a);
  } else {
    if (masked) mhsa_small_kernel<DT, false, true><<<grid, block, shm, st>>>(a);
    else mhsa_small_kernel<DT, false, false><<<grid, block, shm, st>>>(a);
  }
  return folx_launch_status();
}

template <int NW, int DT>
int launch_mhsa(hipStream_t st, const MhsaArgs& a) {
  const int64_t blocks = a.B * a.H;
  if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
  const bool fast = a.n == 16 * NW && a.d == 16 * DT && a.mask == nullptr && a.imask == nullptr;
  const dim3 grid((unsigned)blocks), block(FOLX_WAVE * NW);
  if (a.e != nullptr) {
    if (fast) mhsa_kernel<NW, DT, true, true><<<grid, block, 0, st>>>(a);
    else mhsa_kernel<NW, DT, true, false><<<grid, block, 0, st>>>(a);
  } else {
    if (fast) mhsa_kernel<NW, DT, false, true><<<grid, block, 0, st>>>(a);
    else mhsa_kernel<NW, DT, false, false><<<grid, block, 0, st>>>(a);
  }
  return folx_launch_status();
}

template <int NW>
int launch_mhsa_d(hipStream_t st, const MhsaArgs& a) {
  const int dt = (a.d + 15) / 16;
  switch (dt) {
    case 1: return launch_mhsa<NW, 1>(st, a);
    case 2: return launch_mhsa<NW, 2>(st, a);
    case 3: return launch_mhsa<NW, 3>(st, a);
    default: return launch_mhsa<NW, 4>(st, a);
  }
}

}  // namespace

static int mhsa_entry(void* stream, const float* q, const float* q_jac, const float* q_lap,
                      const float* k, const float* k_jac, const float* k_lap, const float* v,
                      const float* v_jac, const float* v_lap, const float* e, const float* e_jac,
                      const float* e_lap, const uint8_t* mask, const uint8_t* input_mask, float* o,
                      float* o_jac, float* o_lap, int64_t B, int32_t n, int32_t H, int32_t d,
                      int32_t P) {
  if (B < 0 || n <= 0 || H <= 0 || d <= 0 || P < 0) return FOLX_HIP_EINVAL;
  if (B == 0) return FOLX_HIP_OK;
  if (!q || !q_lap || !k || !k_lap || !v || !v_lap || !o || !o_lap) return FOLX_HIP_EINVAL;
  if (P > 0 && (!q_jac || !k_jac || !v_jac || !o_jac)) return FOLX_HIP_EINVAL;
  if (e != nullptr && (!e_lap || (P > 0 && !e_jac))) return FOLX_HIP_EINVAL;
  if (n > 64 || d > 64 || d % 4 != 0) return FOLX_HIP_ENOTSUP;
  const float* ptrs[] = {q, q_jac, q_lap, k, k_jac, k_lap, v, v_jac, v_lap};
  for (const float* p : ptrs)
    if (p && !folx_aligned16(p)) return FOLX_HIP_ENOTSUP;
  MhsaArgs a{q, q_jac, q_lap, k, k_jac, k_lap, v, v_jac, v_lap, e, e_jac, e_lap, mask, input_mask,
             o, o_jac, o_lap, B, n, H, d, P};
  hipStream_t st = (hipStream_t)stream;
  const int nw = (n + 15) / 16;
  switch (nw) {
    case 1:
      // The buffer descriptors of the small form span a walker's (n, H, d) and (n, H, n) blocks with 32-bit offsets, and
      // beyond 16 features it stores two or four floats at a time; mhsa_kernel stores single ones.
      if ((int64_t)n * H * (e && n > d ? n : d) * 4 >= (int64_t)FAR ||
          (d > 16 && !(folx_aligned16(o) && folx_aligned16(o_jac) && folx_aligned16(o_lap))))
        return launch_mhsa_d<2>(st, a);
      switch ((d + 15) / 16) {
        case 1: return launch_mhsa_small<1>(st, a);
        case 2: return launch_mhsa_small<2>(st, a);
        default: return launch_mhsa_small<4>(st, a);
      }
    case 2: return launch_mhsa_d<2>(st, a);
    case 3: return launch_mhsa_d<3>(st, a);
    default: return launch_mhsa_d<4>(st, a);
  }
}

extern "C" int folx_hip_mhsa_fwdlap(void* stream, const float* q, const float* q_jac,
                                    const float* q_lap, const float* k, const float* k_jac,
                                    const float* k_lap, const float* v, const float* v_jac,
                                    const float* v_lap, const uint8_t* mask,
                                    const uint8_t* input_mask, float* o, float* o_jac, float* o_lap,
                                    int64_t B, int32_t n, int32_t H, int32_t d, int32_t P) {
  return mhsa_entry(stream, q, q_jac, q_lap, k, k_jac, k_lap, v, v_jac, v_lap, nullptr, nullptr, nullptr,
                    mask, input_mask, o, o_jac, o_lap, B, n, H, d, P);
}

extern "C" int folx_hip_mhsea_fwdlap(void* stream, const float* q, const float* q_jac,
                                     const float* q_lap, const float* k, const float* k_jac,
                                     const float* k_lap, const float* e, const float* e_jac,
                                     const float* e_lap, const float* v, const float* v_jac,
                                     const float* v_lap, const uint8_t* mask,
                                     const uint8_t* input_mask, float* o, float* o_jac, float* o_lap,
                                     int64_t B, int32_t n, int32_t H, int32_t d, int32_t P) {
  if (!e) return FOLX_HIP_EINVAL;
  return mhsa_entry(stream, q, q_jac, q_lap, k, k_jac, k_lap, v, v_jac, v_lap, e, e_jac, e_lap, mask,
                    input_mask, o, o_jac, o_lap, B, n, H, d, P);
}
