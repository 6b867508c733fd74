// Fused LayerNorm rule over the last axis:  y = g * (x - mean) * rsqrt(var + eps) + beta.
//
// With c = x - mean(x), r = rsqrt(mean(c^2) + eps) and, per Jacobian row u = jac[p],
//   a_p = mean(u),  b_p = mean(c u),  s_p = mean(u^2) - a_p^2
// the triplet of y is
//   y_jac[p] = g r (u - a_p - c r^2 b_p)
//   y_lap    = g r (lap - mean(lap) - c r^2 mean(c lap))                      (linear part)
//            + g ( -2 r^3 sum_p b_p (u_p - a_p) + c (3 r^5 sum_p b_p^2 - r^3 sum_p s_p) )
// which is what the chain mean / sub / square / mean / rsqrt / mul of elementwise and
// reduction rules evaluates to.  A workgroup of 4 wavefronts owns one row of F features and
// streams its Jacobian rows once (read once, written once: 8 (P + 2) F bytes per row, HBM
// bound): wavefront w takes the Jacobian rows p = w, w + 4, ..., four of them in flight at a
// time, so consecutive workgroups walk consecutive addresses of every Jacobian row.  The
// three per-row means are butterfly reductions inside the wavefront; the sums over p meet
// in LDS and wavefront 0 writes y and y_lap.
#include "common.h"

namespace {

__device__ __forceinline__ void wave_sum3(float& a, float& b, float& c) {
#pragma unroll
  for (int off = FOLX_WAVE / 2; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, FOLX_WAVE);
    b += __shfl_xor(b, off, FOLX_WAVE);
    c += __shfl_xor(c, off, FOLX_WAVE);
  }
}
__device__ __forceinline__ float wave_sum1(float a) {
#pragma unroll
  for (int off = FOLX_WAVE / 2; off > 0; off >>= 1) a += __shfl_xor(a, off, FOLX_WAVE);
  return a;
}

// Sums over LW lanes.  Below a wavefront: quad permutes, the two mirrors (which meet equal values in every quad, every half of
// 8 by then) and a swap of neighbouring rows of 16, all vector instructions, where a shuffle is a trip through LDS.
template <int CTRL>
__device__ __forceinline__ float ln_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int LW>
__device__ __forceinline__ float group_sum(float v) {
  if constexpr (LW == FOLX_WAVE) {
    return wave_sum1(v);
  } else {
    v += ln_dpp<0xB1>(v);   // quad_perm [1, 0, 3, 2]
    v += ln_dpp<0x4E>(v);   // quad_perm [2, 3, 0, 1]
    v += ln_dpp<0x141>(v);  // row_half_mirror
    if constexpr (LW > 8) v += ln_dpp<0x140>(v);  // row_mirror
    if constexpr (LW > 16) {
      const auto both = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
      v = __uint_as_float(both[0]) + __uint_as_float(both[1]);
    }
    return v;
  }
}
template <int LW>
__device__ __forceinline__ void group_sum3(float& a, float& b, float& c) {
  if constexpr (LW == FOLX_WAVE) {
    wave_sum3(a, b, c);
  } else {
    a = group_sum<LW>(a); b = group_sum<LW>(b); c = group_sum<LW>(c);
  }
}

constexpr int PSPLIT = 4;

// PER_WAVE: for a few Jacobian rows (sparse storage, P <= 8) a whole workgroup per row of features would
// mostly wait at its barrier: each WAVEFRONT owns a row of features then and walks all P Jacobian rows
// itself (four in flight), no LDS and no barrier.
// LW < 64 lanes to a row of features (F <= 4 LW): the wavefront holds 64 / LW consecutive rows side by side, so that it reads
// and writes up to 1 KB of a Jacobian row at a time whatever F is.  With one row to a wavefront F = 64 left three quarters of
// the lanes idle.  us, one row -> 64 / LW rows: 8192 rows, P = 48: F = 32 85 -> 20, 64 87 -> 41 (5.2 TB/s), 96 91 -> 60,
// 128 95 -> 82; 1000 rows, P = 96, F = 64: 27 -> 13.5; 32 768 rows, P = 3, F = 64: 42 -> 17; 100 rows, P = 12: 5.6 -> 4.8.
template <int NV, bool PER_WAVE, int LW = FOLX_WAVE>
__global__ __launch_bounds__(FOLX_WAVE * PSPLIT) void layernorm_kernel(
    const float* __restrict__ x, const float* __restrict__ jac, const float* __restrict__ lap,
    const float* __restrict__ gamma, const float* __restrict__ beta, float* __restrict__ y,
    float* __restrict__ y_jac, float* __restrict__ y_lap, int64_t R, int32_t F, int32_t P, float eps) {
  __shared__ float4 redT[PSPLIT][NV * FOLX_WAVE];
  constexpr int ROWS = FOLX_WAVE / LW;  // of features, per wavefront
  __shared__ float reds[PSPLIT][ROWS][2];
  const int wlane = threadIdx.x % FOLX_WAVE;
  const int lane = wlane % LW, sub = wlane / LW;
  const int w = threadIdx.x / FOLX_WAVE;
  const int64_t first = (PER_WAVE ? (int64_t)blockIdx.x * PSPLIT + w : (int64_t)blockIdx.x) * ROWS;
  if (PER_WAVE && first >= R) return;
  const bool live = ROWS == 1 || first + sub < R;
  const int64_t row = live ? first + sub : R - 1;
  constexpr int PS = PER_WAVE ? 1 : PSPLIT;  // distance between the Jacobian rows of a wavefront
  const int F4 = F / 4;
  const float invF = 1.0f / (float)F;
  const int64_t S = R * (int64_t)F;  // elements per Jacobian row
  const int64_t off = row * (int64_t)F;

  bool ok[NV];
  float4 c[NV], g[NV];
  float sx = 0.0f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i4 = lane + LW * v;
    ok[v] = live && i4 < F4;
    c[v] = make_float4(0.f, 0.f, 0.f, 0.f);
    g[v] = c[v];
    if (ok[v]) {
      c[v] = *reinterpret_cast<const float4*>(x + off + 4 * i4);
      g[v] = gamma ? *reinterpret_cast<const float4*>(gamma + 4 * i4) : make_float4(1.f, 1.f, 1.f, 1.f);
      sx += c[v].x + c[v].y + c[v].z + c[v].w;
    }
  }
  const float mu = group_sum<LW>(sx) * invF;
  float sv = 0.0f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (ok[v]) {
      c[v].x -= mu; c[v].y -= mu; c[v].z -= mu; c[v].w -= mu;
      sv += c[v].x * c[v].x + c[v].y * c[v].y + c[v].z * c[v].z + c[v].w * c[v].w;
    }
  }
  const float var = group_sum<LW>(sv) * invF;
  const float r = 1.0f / sqrtf(var + eps);
  const float r2 = r * r, r3 = r2 * r, r5 = r3 * r2;

  float4 T[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) T[v] = make_float4(0.f, 0.f, 0.f, 0.f);
  float sb2 = 0.0f, ss = 0.0f;

  auto load_row = [&](int p, float4* u) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      u[v] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (ok[v]) u[v] = folx_ld_stream4(jac + (int64_t)p * S + off + 4 * (lane + LW * v));
    }
  };
  auto partial = [&](const float4* u, float& s1, float& s2, float& s3) {
    s1 = s2 = s3 = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      s1 += u[v].x + u[v].y + u[v].z + u[v].w;
      s2 += c[v].x * u[v].x + c[v].y * u[v].y + c[v].z * u[v].z + c[v].w * u[v].w;
      s3 += u[v].x * u[v].x + u[v].y * u[v].y + u[v].z * u[v].z + u[v].w * u[v].w;
    }
  };
  auto finish_row = [&](int p, const float4* u, float s1, float s2, float s3) {
    const float a = s1 * invF, b = s2 * invF;
    sb2 += b * b;
    ss += s3 * invF - a * a;
    const float cb = r2 * b;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (ok[v]) {
        const float dx = u[v].x - a, dy = u[v].y - a, dz = u[v].z - a, dw = u[v].w - a;
        T[v].x += b * dx; T[v].y += b * dy; T[v].z += b * dz; T[v].w += b * dw;
        float4 o;
        o.x = g[v].x * r * (dx - c[v].x * cb);
        o.y = g[v].y * r * (dy - c[v].y * cb);
        o.z = g[v].z * r * (dz - c[v].z * cb);
        o.w = g[v].w * r * (dw - c[v].w * cb);
        folx_st_stream4(y_jac + (int64_t)p * S + off + 4 * (lane + LW * v), o);
      }
    }
  };

  int p = PER_WAVE ? 0 : w;
  for (; p + 3 * PS < P; p += 4 * PS) {  // four Jacobian rows in flight per wavefront
    float4 u0[NV], u1[NV], u2[NV], u3[NV];
    load_row(p, u0);
    load_row(p + PS, u1);
    load_row(p + 2 * PS, u2);
    load_row(p + 3 * PS, u3);
    float a1, a2, a3, b1, b2, b3, c1, c2, c3, e1, e2, e3;
    partial(u0, a1, a2, a3);
    partial(u1, b1, b2, b3);
    partial(u2, c1, c2, c3);
    partial(u3, e1, e2, e3);
    group_sum3<LW>(a1, a2, a3);
    group_sum3<LW>(b1, b2, b3);
    group_sum3<LW>(c1, c2, c3);
    group_sum3<LW>(e1, e2, e3);
    finish_row(p, u0, a1, a2, a3);
    finish_row(p + PS, u1, b1, b2, b3);
    finish_row(p + 2 * PS, u2, c1, c2, c3);
    finish_row(p + 3 * PS, u3, e1, e2, e3);
  }
  for (; p < P; p += PS) {
    float4 u0[NV];
    load_row(p, u0);
    float a1, a2, a3;
    partial(u0, a1, a2, a3);
    group_sum3<LW>(a1, a2, a3);
    finish_row(p, u0, a1, a2, a3);
  }

  // the sums over p of the four wavefronts meet in LDS (this barrier also orders every
  // wavefront's read of x before the write of y, which makes in-place use safe)
  if constexpr (!PER_WAVE) {
#pragma unroll
    for (int v = 0; v < NV; ++v) redT[w][v * FOLX_WAVE + wlane] = T[v];
    if (lane == 0) { reds[w][sub][0] = sb2; reds[w][sub][1] = ss; }
    __syncthreads();
    if (w != 0) return;
    sb2 = reds[0][sub][0]; ss = reds[0][sub][1];
#pragma unroll
    for (int ww = 1; ww < PSPLIT; ++ww) {
      sb2 += reds[ww][sub][0]; ss += reds[ww][sub][1];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const float4 t = redT[ww][v * FOLX_WAVE + wlane];
        T[v].x += t.x; T[v].y += t.y; T[v].z += t.z; T[v].w += t.w;
      }
    }
  }

  // value and Laplacian
  float4 l[NV];
  float sl = 0.0f, scl = 0.0f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    l[v] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (ok[v]) {
      l[v] = *reinterpret_cast<const float4*>(lap + off + 4 * (lane + LW * v));
      sl += l[v].x + l[v].y + l[v].z + l[v].w;
      scl += c[v].x * l[v].x + c[v].y * l[v].y + c[v].z * l[v].z + c[v].w * l[v].w;
    }
  }
  float dummy = 0.0f;
  group_sum3<LW>(sl, scl, dummy);
  const float ml = sl * invF, mcl = scl * invF;
  const float k2 = 3.0f * r5 * sb2 - r3 * ss;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (ok[v]) {
      const int i4 = lane + LW * v;
      const float4 bt = beta ? *reinterpret_cast<const float4*>(beta + 4 * i4) : make_float4(0.f, 0.f, 0.f, 0.f);
      float4 yo, lo;
      yo.x = g[v].x * r * c[v].x + bt.x; yo.y = g[v].y * r * c[v].y + bt.y;
      yo.z = g[v].z * r * c[v].z + bt.z; yo.w = g[v].w * r * c[v].w + bt.w;
      lo.x = g[v].x * (r * (l[v].x - ml - c[v].x * r2 * mcl) - 2.0f * r3 * T[v].x + c[v].x * k2);
      lo.y = g[v].y * (r * (l[v].y - ml - c[v].y * r2 * mcl) - 2.0f * r3 * T[v].y + c[v].y * k2);
      lo.z = g[v].z * (r * (l[v].z - ml - c[v].z * r2 * mcl) - 2.0f * r3 * T[v].z + c[v].z * k2);
      lo.w = g[v].w * (r * (l[v].w - ml - c[v].w * r2 * mcl) - 2.0f * r3 * T[v].w + c[v].w * k2);
      *reinterpret_cast<float4*>(y + off + 4 * i4) = yo;
      *reinterpret_cast<float4*>(y_lap + off + 4 * i4) = lo;
    }
  }
}

}  // namespace

extern "C" int folx_hip_layernorm_fwdlap(void* stream, const float* x, const float* jac,
                                         const float* lap, const float* gamma, const float* beta,
                                         float* y, float* y_jac, float* y_lap, int64_t R, int32_t F,
                                         int32_t P, float eps) {
  if (R < 0 || F <= 0 || P < 0) return FOLX_HIP_EINVAL;
  if (R == 0) return FOLX_HIP_OK;
  if (!x || !lap || !y || !y_lap || (P > 0 && (!jac || !y_jac))) return FOLX_HIP_EINVAL;
  if (F % 4 != 0 || F > 1024) return FOLX_HIP_ENOTSUP;
  const void* ptrs[] = {x, jac, lap, gamma, beta, y, y_jac, y_lap};
  for (const void* p : ptrs)
    if (p && !folx_aligned16(p)) return FOLX_HIP_ENOTSUP;
  const bool per_wave = P <= 8;
  const int lw = F <= 32 ? 8 : (F <= 64 ? 16 : (F <= 128 ? 32 : FOLX_WAVE));
  const int64_t rows = (int64_t)(FOLX_WAVE / lw) * (per_wave ? PSPLIT : 1);  // of features, per workgroup
  const int64_t blocks = (R + rows - 1) / rows;
  if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)blocks), block(FOLX_WAVE * PSPLIT);
  const int nv = (F / 4 + FOLX_WAVE - 1) / FOLX_WAVE;
#define FOLX_LN(NV, LW)                                                                                               \
  if (per_wave) layernorm_kernel<NV, true, LW><<<grid, block, 0, st>>>(x, jac, lap, gamma, beta, y, y_jac, y_lap, R, F, P, eps); \
  else layernorm_kernel<NV, false, LW><<<grid, block, 0, st>>>(x, jac, lap, gamma, beta, y, y_jac, y_lap, R, F, P, eps);
  switch (lw < FOLX_WAVE ? -lw : nv) {
    case -8: FOLX_LN(1, 8) break;
    case -16: FOLX_LN(1, 16) break;
    case -32: FOLX_LN(1, 32) break;
    case 1: FOLX_LN(1, FOLX_WAVE) break;
    case 2: FOLX_LN(2, FOLX_WAVE) break;
    case 3: FOLX_LN(3, FOLX_WAVE) break;
    default: FOLX_LN(4, FOLX_WAVE) break;
  }
#undef FOLX_LN
  return folx_launch_status();
}
