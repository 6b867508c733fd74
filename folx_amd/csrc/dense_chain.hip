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
// returns the bits of its layers run one by one.  Inside a run of 16 k the tile is stored in the order in which the lanes take
// it, so that they read 128 bits at a time.
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

// W[k][col] for the four k of this lane in chunk j (16 k); past K zero
__device__ __forceinline__ void chain_weights(const ChainLayer& ly, int col, int lq, int j, float (&w)[4]) {
  const int c = min(col, ly.N - 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = 16 * j + 8 * (i / 2) + 4 * (lq & 1) + 2 * (i % 2) + (lq >> 1);
    const float v = ly.W[min(k, ly.K - 1) * ly.N + c];
    w[i] = k < ly.K ? v : 0.f;
  }
}

template <int NR, int PB>
__global__ __launch_bounds__(512, 4) void dense_chain_kernel(ChainParams a) {
  constexpr bool HALF = PB == 8;
  constexpr int NB = HALF ? (NR + 1) / 2 : NR;
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
  chain_weights(a.layer[0], col, lq, 0, wA);
  chain_weights(a.layer[0], col, lq, 1, wB);

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
      auto chunk = [&](int j, float (&w)[4]) __attribute__((always_inline)) {
        floatx4 v[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) v[b] = *reinterpret_cast<const floatx4*>(base + b * bs + 16 * j);
        const float wv[4] = {w[0], w[1], w[2], w[3]};
        chain_weights(ly, col, lq, j + 2, w);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i], v[b][i], acc[b], 0, 0, 0);
      };
      for (int j = 0; j < chunks; j += 2) {
        chunk(j, wA);
        if (j + 1 < chunks) chunk(j + 1, wB);
      }
    }
    const bool last = l + 1 == L;
    const bool store = last || (l + 2 == L && a.h != nullptr);
    if (!last) {
      chain_weights(a.layer[l + 1], col, lq, 0, wA);
      chain_weights(a.layer[l + 1], col, lq, 1, wB);
    }
    if (active) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float o, d1, d2, ssq = 0.f;
        if constexpr (HALF) {
          const float zo = other_half(acc[0][r]);
          act_eval_fused(ly.act, (half == 0 ? acc[0][r] : zo) + bias[r], ly.prm, o, d1, d2);
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
        } else {
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
  pl.pb = (R + 15) / 16 <= 256 ? 8 : 16;
  const int nr = P + 2, nb = pl.pb == 8 ? (nr + 1) / 2 : nr;
  pl.lds = (int64_t)nb * 16 * pl.ld * 4;
  pl.blocks = (R + pl.pb - 1) / pl.pb;
  return pl.blocks <= 0x7fffffffLL;
}

template <int NR, int PB>
int launch_chain(hipStream_t st, const ChainParams& prm, const ChainPlan& pl) {
  if (pl.lds > 65536 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(&dense_chain_kernel<NR, PB>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds) != hipSuccess)
    return FOLX_HIP_ELAUNCH;
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
  return L > 1 && plan_chain(L, act, widths, R, P, pl) ? 1 : 0;
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
