// A chain of narrow dense + activation layers (K, N <= 128) in one launch, with few Jacobian rows (P <= 6):
//   z = x @ W + bias      x   <- f(z)
//   zj[p] = jac[p] @ W    jac <- f'(z) zj
//   zl = lap @ W          lap <- f'(z) zl + f''(z) sum_p zj[p]^2         layer by layer,
// optionally ending in a matrix-vector product (N = 1, no activation).
//
// Layer by layer, such a network moves its triplet through memory between every two layers and, on a small batch, pays one
// load, one product and one store in sequence per layer.  Here a workgroup owns PB positions, keeps all P + 2 rows of their
// triplet in LDS from the first layer to the last, and only the weights of each layer (40 KB at 100 x 100, from L2) come in
// between.  Wavefront w forms columns 16 w .. 16 w + 15 of every row of the triplet side by side (v_mfma_f32_16x16x4_f32, the
// product transposed: a lane holds 4 consecutive columns of one position), which leaves f', f'' and the sum over Jacobian
// rows as register arithmetic, and writes its output over the input tile between two barriers that wait for LDS only: the
// first weights of the next layer are asked for before them.
//
// LDS tile: [block][16 rows][ld] floats, ld = 4 (mod 8).  PB = 16: block s holds row s of the triplet.  PB = 8: block b holds
// rows 2 b and 2 b + 1 of the triplet, 8 positions each, so that a small batch spreads over twice the workgroups; the lanes of
// one half take what they need from the other by a rotation inside 16 lanes.
// A column's products are added in the order of dense_act.hip (two of its steps in one instruction: k = 8 j + 4 (q % 2) +
// 2 e + q / 2 for lane group q of step e), and the matrix-vector product at the end in that of dense_n1_flat_kernel, so a chain
// returns the bits of its layers run one by one in dense_act_few_kernel (the general kernel rounds d1 z_lap + d2 ssq the other
// way round).  Inside a run of 16 k the tile is stored in the order in which the lanes take it, so that they read 128 bits at a
// time.
//
// What bounds it: the matrix pipe together with the other instructions of its wavefronts (442 vector instructions a layer and
// wavefront beside 156 matrix ones at 100 x 100, P = 4; the pipe busy 47 % of the time, and 16 % of the time CUs without work at
// the end), and for 100 features the four SIMDs' unequal shares of seven wavefronts: 70 TFLOP/s there, 100 at 128 x 128, P = 6.
// Weights through a descriptor and operands one chunk ahead: 8 to 14 % of the time.  80 registers for a third workgroup a
// CU spilled 70 of them (429 -> 631 us).  us, layers one by one -> chain: ten layers of 100, P = 4: 2000 positions
// 101 -> 43, 25 600 503 -> 390; four of 50, P = 3, 15 750: 106 -> 31; six of 128, P = 6, 100 000: 1408 -> 1156.
#include "activations.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int MAXL = FOLX_HIP_CHAIN_MAX_LAYERS;
constexpr int MAXP = 6;

struct ChainLayer {
  const float *W, *bias;
  int32_t K, N, act;  // act < 0: none (last layer, N = 1)
  float prm;
};

struct ChainParams {
  const float *x, *jac, *lap;
  float *y, *y_jac, *y_lap;
  float *h, *h_jac, *h_lap;  // what goes into a matrix-vector product at the end, where somebody else reads it too
  int64_t R;
  int32_t P, L, ld, vec;
  ChainLayer layer[MAXL];
};

// where feature k of a row is kept
__device__ __forceinline__ int chain_slot(int k) {
  return (k & ~15) + 4 * (((k >> 2) & 1) + 2 * (k & 1)) + 2 * ((k >> 3) & 1) + ((k >> 1) & 1);
}

// LDS traffic of this workgroup is complete; weights on their way stay on their way
__device__ __forceinline__ void chain_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// the value of the lane 8 further on in its group of 16
__device__ __forceinline__ float other_half(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));
}

// A lane's weights of one column: chunk j (16 k) gives it k = 16 j + 4 (lq % 2) + lq / 2 + {0, 2, 8, 10}.  Loads through a
// descriptor of the K N floats, chunk after chunk: past K they bring zero.  (Past N, too wide a wavefront's columns are those
// of the next row: never stored.)
struct ChainW {
  __amdgpu_buffer_rsrc_t rsrc;
  int chunk;   // bytes from one chunk to the next
  int off[4];  // bytes, of the next chunk
  __device__ __forceinline__ void layer(const ChainLayer& ly, int col, int lq) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ly.W), 0, ly.K * ly.N * 4, 0x00027000);
    chunk = 64 * ly.N;
    const int k0 = 4 * (lq & 1) + (lq >> 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) off[i] = 4 * ((k0 + 8 * (i / 2) + 2 * (i % 2)) * ly.N + col);
  }
  __device__ __forceinline__ void next(float (&w)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off[i], 0, 0));
      off[i] += chunk;
    }
  }
};

template <int NR, int PB>
__global__ __launch_bounds__(512, 4) void dense_chain_kernel(ChainParams a) {
  constexpr bool HALF = PB == 8;
  constexpr int NB = HALF ? (NR + 1) / 2 : NR;
  constexpr bool AHEAD = NB <= 6;  // operands from LDS one chunk ahead of their products: 4 NB registers, and 128 are to be had
  extern __shared__ __attribute__((aligned(16))) float tile[];
  const int tid = threadIdx.x;
  const int nthr = blockDim.x;
  const int lane = tid % 64;
  const int wave = folx_wave_id();
  const int l16 = lane % 16, lq = lane / 16;
  const int half = HALF ? l16 / 8 : 0;
  const int64_t R = a.R;
  const int64_t r0 = (int64_t)blockIdx.x * PB;
  const int ld = a.ld, bs = 16 * ld;
  const int last_pos = (int)(R - 1 - r0 < PB - 1 ? R - 1 - r0 : PB - 1);
  const int col = 16 * wave + l16;  // as the product's W operand

  float wA[4], wB[4];
  ChainW weights;
  weights.layer(a.layer[0], col, lq);
  weights.next(wA);
  weights.next(wB);

  {  // the input triplet, zero from K to the next multiple of 16
    const int K = a.layer[0].K, Kp = (K + 15) / 16 * 16;
    const int64_t RK = R * K;
    for (int f = tid; f < PB * Kp; f += nthr) {
      const int m = f / Kp, k = f - m * Kp;
      const int64_t at = (r0 + min(m, last_pos)) * K + min(k, K - 1);
      float v[NR];
#pragma unroll
      for (int s = 0; s < NR; ++s) v[s] = (s == 0 ? a.x : (s < NR - 1 ? a.jac + (s - 1) * RK : a.lap))[at];
      float* to = tile + m * ld + chain_slot(k);
#pragma unroll
      for (int s = 0; s < NR; ++s) to[HALF ? s / 2 * bs + s % 2 * 8 * ld : s * bs] = k < K ? v[s] : 0.f;
      if constexpr (HALF && NR % 2 == 1) to[(NB - 1) * bs + 8 * ld] = 0.f;
    }
  }
  chain_barrier();

  const int L = a.L;
  for (int l = 0; l < L; ++l) {
    const ChainLayer ly = a.layer[l];
    const int K = ly.K, N = ly.N;
    if (ly.act < 0) {
      // one thread per row of the triplet: K / 4 partial products of four, even and odd ones added up separately
      const int K4 = (K + 3) / 4;
      for (int i = tid; i < NR * PB; i += nthr) {
        const int s = i / PB, m = i % PB;
        if (m > last_pos) continue;
        const float* row = tile + (HALF ? s / 2 * bs + (m + s % 2 * 8) * ld : s * bs + m * ld);
        float sum[2] = {0.f, 0.f};
        for (int c = 0; c < K4; ++c) {
          const float* q = row + (c / 4) * 16 + 4 * (c % 2) + 2 * (c / 2 % 2);  // k = 4 c, 4 c + 2; 8 further on 4 c + 1, 4 c + 3
          const float w0 = ly.W[4 * c], w1 = 4 * c + 1 < K ? ly.W[4 * c + 1] : 0.f;
          const float w2 = 4 * c + 2 < K ? ly.W[4 * c + 2] : 0.f, w3 = 4 * c + 3 < K ? ly.W[4 * c + 3] : 0.f;
          const float part = fmaf(q[0], w0, fmaf(q[8], w1, fmaf(q[1], w2, q[9] * w3)));
          if (c & 1) sum[1] += part; else sum[0] += part;
        }
        const float o = sum[0] + sum[1] + (s == 0 && ly.bias != nullptr ? ly.bias[0] : 0.f);
        (s == 0 ? a.y : (s < NR - 1 ? a.y_jac + (s - 1) * R : a.y_lap))[r0 + m] = o;
      }
      return;
    }
    const bool active = 16 * wave < N;
    const int n0 = 16 * wave + 4 * lq;  // first of this lane's four columns of the result
    floatx4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (active) {
      if (ly.bias != nullptr) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[r] = ly.bias[min(n0 + r, N - 1)];
      }
      const int chunks = (K + 15) / 16;
      const float* base = tile + l16 * ld + 4 * lq;
      floatx4 vA[NB], vB[NB];
      auto read = [&](int j, floatx4 (&v)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b) v[b] = *reinterpret_cast<const floatx4*>(base + b * bs + 16 * j);
      };
      // the products of chunk j, while chunk j + 1 comes from LDS and the weights of chunk j + 2 from memory
      auto chunk = [&](int j, float (&w)[4], floatx4 (&v)[NB], floatx4 (&next)[NB]) __attribute__((always_inline)) {
        if constexpr (AHEAD) {
          if (j + 1 < chunks) read(j + 1, next);
        } else {
          read(j, v);
        }
        const float wv[4] = {w[0], w[1], w[2], w[3]};
        weights.next(w);
        if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i], v[b][i], acc[b], 0, 0, 0);
        if (16 * j + 8 < K)
#pragma unroll
          for (int i = 2; i < 4; ++i)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i], v[b][i], acc[b], 0, 0, 0);
      };
      if constexpr (AHEAD) read(0, vA);
      for (int j = 0; j < chunks; j += 2) {
        chunk(j, wA, vA, AHEAD ? vB : vA);
        if (j + 1 < chunks) chunk(j + 1, wB, AHEAD ? vB : vA, vA);
      }
    }
    const bool last = l + 1 == L;
    const bool store = last || (l + 2 == L && a.h != nullptr);
    if (!last) {
      weights.layer(a.layer[l + 1], col, lq);
      weights.next(wA);
      weights.next(wB);
    }
    if (active) {
      if constexpr (HALF) {
        // rows 2 b and 2 b + 1 of the triplet are in the two halves of a group of 16 lanes: one half evaluates the function of
        // columns 0 and 2, the other that of 1 and 3, and they exchange the results
#pragma unroll
        for (int r2 = 0; r2 < 4; r2 += 2) {
          const float z0 = acc[0][r2], z1 = other_half(acc[0][r2 + 1]);  // half 0: column r2; half 1: column r2 + 1
          float e, e1, e2;
          act_eval_fused(ly.act, (half == 0 ? z0 : z1) + (half == 0 ? bias[r2] : bias[r2 + 1]), ly.prm, e, e1, e2);
          const float f = other_half(e), f1 = other_half(e1), f2 = other_half(e2);
#pragma unroll
          for (int r = r2; r < r2 + 2; ++r) {
            const bool own = half == r - r2;
            const float o = own ? e : f, d1 = own ? e1 : f1, d2 = own ? e2 : f2;
            float ssq = 0.f;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              const float mine = acc[b][r], theirs = other_half(mine);
              const float lo = half == 0 ? mine : theirs, hi = half == 0 ? theirs : mine;
              if (b > 0 && 2 * b < NR - 1) ssq += lo * lo;
              if (2 * b + 1 < NR - 1) ssq += hi * hi;
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              const float v = d1 * acc[b][r];
              const float with_lap = d1 * acc[b][r] + d2 * ssq;
              // row of the triplet: 2 b (half 0) or 2 b + 1
              const float lo = b == 0 ? o : (2 * b == NR - 1 ? with_lap : v);
              const float hi = 2 * b + 1 == NR - 1 ? with_lap : v;
              acc[b][r] = half == 0 ? lo : hi;
            }
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float o, d1, d2, ssq = 0.f;
          act_eval_fused(ly.act, acc[0][r] + bias[r], ly.prm, o, d1, d2);
          acc[0][r] = o;
#pragma unroll
          for (int s = 1; s < NR - 1; ++s) {
            ssq += acc[s][r] * acc[s][r];
            acc[s][r] *= d1;
          }
          acc[NR - 1][r] = d1 * acc[NR - 1][r] + d2 * ssq;
        }
      }
    }
    if (store) {
      const int m = HALF ? l16 % 8 : l16;
      const int cols = min(4, N - n0);
      if (active && m <= last_pos && cols > 0) {
        float *const out = last ? a.y : a.h, *const out_jac = last ? a.y_jac : a.h_jac, *const out_lap = last ? a.y_lap : a.h_lap;
        const int64_t at = (r0 + m) * N + n0, RN = R * N;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int s = HALF ? 2 * b + half : b;
          if (HALF && s >= NR) break;
          float* p = (s == 0 ? out : (s < NR - 1 ? out_jac + (s - 1) * RN : out_lap)) + at;
          if (a.vec) *reinterpret_cast<floatx4*>(p) = acc[b];
          else
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (r < cols) p[r] = acc[b][r];
        }
      }
      if (last) return;
    }
    chain_barrier();  // every wavefront has read the tile
    if (active) {
      // columns 4 lq + r of a run of 16: (0, 2) and (1, 3) lie side by side.  Columns past N are written as zeros: they meet
      // zeros of the next W.
      float* to = tile + l16 * ld + 16 * wave + 4 * (lq & 1) + 2 * (lq >> 1);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        floatx4 v = acc[b];
        if (16 * wave + 16 > N)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = n0 + r < N ? v[r] : 0.f;
        *reinterpret_cast<float2*>(to + b * bs) = make_float2(v[0], v[2]);
        *reinterpret_cast<float2*>(to + b * bs + 8) = make_float2(v[1], v[3]);
      }
    }
    chain_barrier();
  }
}

struct ChainPlan {
  int waves, ld, pb;
  int64_t blocks, lds;
};

// false: not a chain this file is built for
bool plan_chain(int32_t L, const int32_t* act, const int32_t* widths, int64_t R, int32_t P, ChainPlan& pl) {
  if (L < 1 || L > MAXL || P > MAXP) return false;
  int kmax = 0, nmax = 0;
  for (int l = 0; l < L; ++l) {
    const int K = widths[l], N = widths[l + 1];
    if (K > 128 || N > 128) return false;
    if (act[l] < 0 ? (l + 1 < L || N != 1) : !act_fused(act[l])) return false;
    kmax = K > kmax ? K : kmax;
    if (act[l] >= 0) nmax = N > nmax ? N : nmax;
  }
  pl.waves = (nmax + 15) / 16;
  if (pl.waves < 1) pl.waves = 1;
  pl.ld = (kmax + 15) / 16 * 16 + 4;
  // 8 positions give the shorter chain per workgroup, 16 the better use of the weights and fewer idle lanes.  us, 8 / 16: four
  // layers of 100, P = 4: R = 2000 17.9 / 25.8, 3000 27.2 / 26.3, 6000 40.5 / 42.9, 8000 50.8 / 43.6, 50 000 288 / 260; three of 32,
  // P = 6: 2000 8.5 / 10.8, 6000 11.0 / 13.9, 12 000 16.4 / 15.0; three of 128, P = 6: 4100 40.1 / 42.8, 8000 53.8 / 46.5.
  pl.pb = R <= 6144 ? 8 : 16;
  const int nr = P + 2, nb = pl.pb == 8 ? (nr + 1) / 2 : nr;
  pl.lds = (int64_t)nb * 16 * pl.ld * 4;
  pl.blocks = (R + pl.pb - 1) / pl.pb;
  return pl.blocks <= 0x7fffffffLL;
}

// us of the chain and of its layers one by one (multiples of 4 wide): launches, a round of workgroups (per layer, and per chunk of 16
// features and block of rows), MB moved, products; a launch's rows and the columns of its output.  Fitted to 419 chains (2 to 8
// layers of 4 to 128 features, equal, unequal and narrow in the middle, R = 500 .. 320 000, P = 0 .. 6; 12 and 11 % rms; another
// 607: 13 and 12 %).  A chain saves the trips through memory between its layers and nothing at its ends, where its workgroups stream
// worse than those of one layer: 128 -> 4 -> 128 over 200 000 positions, P = 1: 160 us layer by layer, 258 in one; 4000: 13 and 8.7.
// Of the 607, taken whenever they fit, 78 were more than 3 % slower than their layers, up to 2.7 times (0.704 of the layers' time in
// the mean); by this rule 7 are, by at most 13 %, and 17 that
// would gain more than 3 %, up to 25, stay apart (0.690; the faster of both each time: 0.686).
double chain_time(const ChainPlan& pl, int32_t L, const int32_t* widths, int64_t R, int32_t P) {
  const int nr = P + 2, nb = pl.pb == 8 ? (nr + 1) / 2 : nr;
  const int64_t by_lds = (160 << 10) / pl.lds;
  const double per_cu = (double)(by_lds < 16 / pl.waves ? by_lds : 16 / pl.waves);
  double rounds = (double)pl.blocks / (256.0 * per_cu);
  if (rounds < 1.0) rounds = 1.0;
  int chunks = 0, tiles = 0;
  for (int l = 0; l < L; ++l) {
    const int c = (widths[l] + 15) / 16;
    chunks += c;
    tiles += c * ((widths[l + 1] + 15) / 16);
  }
  return 2.3 + rounds * (1.06 * L + 0.094 * nb * chunks) + 0.155 * 4e-6 * (double)R * nr * (widths[0] + widths[L]) +
         53.5e-6 * (double)R / 16 * nr * tiles;
}

double layers_time(int32_t L, const int32_t* widths, int64_t R, int32_t P) {
  const int nr = P + 2;
  double t = 0.0;
  for (int l = 0; l < L; ++l) {
    const int K = widths[l], N = widths[l + 1];
    t += 2.74 + 0.155 * nr + 0.033 * N +
         (double)R * nr * (0.176 * 4e-6 * (K + N) + 13.5e-9 * ((K + 7) / 8 * 8) * ((N + 15) / 16 * 16));
  }
  return t;
}

template <int NR, int PB>
int launch_chain(hipStream_t st, const ChainParams& prm, const ChainPlan& pl) {
  if (pl.lds > 65536) {
    static FolxLdsGrant grant;
    if (!grant.ask(reinterpret_cast<const void*>(&dense_chain_kernel<NR, PB>), 160 * 1024)) return FOLX_HIP_ELAUNCH;
  }
  dense_chain_kernel<NR, PB><<<dim3((unsigned)pl.blocks), dim3(64 * pl.waves), pl.lds, st>>>(prm);
  return folx_launch_status();
}

template <int NR>
int launch_rows(hipStream_t st, const ChainParams& prm, const ChainPlan& pl) {
  return pl.pb == 8 ? launch_chain<NR, 8>(st, prm, pl) : launch_chain<NR, 16>(st, prm, pl);
}

}  // namespace

extern "C" int folx_hip_dense_chain_faster(int32_t L, const int32_t* act, const int32_t* widths, int64_t R, int32_t P) {
  ChainPlan pl;
  if (L < 1 || !act || !widths || R <= 0 || P < 0) return FOLX_HIP_EINVAL;
  if (L < 2 || !plan_chain(L, act, widths, R, P, pl)) return 0;
  // A layer whose input is no multiple of 4 wide is a product and a function on their own, which add in another order: the chain
  // then, for any number of positions (of 174 such chains 5 were slower than their layers, by 8 to 19 %).
  for (int l = 0; l < L; ++l)
    if (widths[l] % 4 != 0) return 1;
  return chain_time(pl, L, widths, R, P) < layers_time(L, widths, R, P) ? 1 : 0;
}

extern "C" int folx_hip_dense_chain_fwdlap(void* stream, int32_t L, const int32_t* act, const float* param,
                                           const float* const* W, const float* const* bias, const int32_t* widths,
                                           const float* x, const float* jac, const float* lap, float* y, float* y_jac,
                                           float* y_lap, float* h, float* h_jac, float* h_lap, int64_t R,
                                           int32_t P) {
  if (L < 1 || !act || !param || !W || !bias || !widths || R < 0 || P < 0) return FOLX_HIP_EINVAL;
  for (int l = 0; l <= L && l <= MAXL; ++l)
    if (widths[l] <= 0 || (l < L && l < MAXL && !W[l])) return FOLX_HIP_EINVAL;
  ChainPlan pl;
  if (!plan_chain(L, act, widths, R, P, pl)) return FOLX_HIP_ENOTSUP;
  if (R == 0) return FOLX_HIP_OK;
  if (!x || !lap || !y || !y_lap || (P > 0 && (!jac || !y_jac))) return FOLX_HIP_EINVAL;
  const bool vector_last = act[L - 1] < 0;
  if ((h != nullptr) != (h_lap != nullptr) || (P > 0 && (h != nullptr) != (h_jac != nullptr)) ||
      (h != nullptr && (!vector_last || L < 2)))
    return FOLX_HIP_EINVAL;
  ChainParams prm;
  prm.x = x; prm.jac = jac; prm.lap = lap;
  prm.y = y; prm.y_jac = y_jac; prm.y_lap = y_lap;
  prm.h = h; prm.h_jac = h_jac; prm.h_lap = h_lap;
  prm.R = R; prm.P = P; prm.L = L; prm.ld = pl.ld;
  // the matrix-vector product stores single floats whatever the alignment
  prm.vec = vector_last ? widths[L - 1] % 4 == 0 && folx_aligned16(h) && folx_aligned16(h_jac) && folx_aligned16(h_lap)
                        : widths[L] % 4 == 0 && folx_aligned16(y) && folx_aligned16(y_jac) && folx_aligned16(y_lap);
  for (int l = 0; l < L; ++l) prm.layer[l] = {W[l], bias[l], widths[l], widths[l + 1], act[l], param[l]};
  hipStream_t st = (hipStream_t)stream;
  switch (P) {
    case 0: return launch_rows<2>(st, prm, pl);
    case 1: return launch_rows<3>(st, prm, pl);
    case 2: return launch_rows<4>(st, prm, pl);
    case 3: return launch_rows<5>(st, prm, pl);
    case 4: return launch_rows<6>(st, prm, pl);
    case 5: return launch_rows<7>(st, prm, pl);
    default: return launch_rows<8>(st, prm, pl);
  }
}
