// Reductions over a middle axis: in [rows][outer][red][inner] -> out [rows][outer][inner].
// The sum rule is linear, so the same kernel serves x, the Jacobian rows and lap.  The
// reduced axis may be a window [lo, hi) of a longer axis (a slice that is summed right away is
// read where it lies): `span` is the full length of that axis in memory.
#include "common.h"

namespace {

// Up to three arrays (a triplet's value, Jacobian rows and Laplacian) in one launch: outputs are numbered through, end[a] is
// the first number behind array a.  On small batches a launch of its own for each cost more than its work (7 electrons, 512
// walkers: a spin-wise mean of the value 4.7 us where its Jacobian rows take 8).
struct Arrays {
  const float* in[3];
  float* out[3];
  int64_t end[3];
  // the array of output o, which becomes its number inside that array
  __device__ __forceinline__ void find(int64_t& o, const float*& src, float*& dst) const {
    src = in[0]; dst = out[0];
    if (o >= end[0]) {
      const bool third = o >= end[1];
      src = third ? in[2] : in[1];
      dst = third ? out[2] : out[1];
      o -= third ? end[1] : end[0];
    }
  }
};

// inner >= 2: one thread per output element, consecutive threads on consecutive `inner`
// positions so every step of the loop over `red` is a coalesced read.
template <bool MAX>
__global__ __launch_bounds__(256) void reduce_mid_kernel(Arrays arrays, int64_t total, int64_t red,
                                                         int64_t inner, int64_t span, int64_t lo, float alpha) {
  int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= total) return;
  const float* in;
  float* out;
  arrays.find(o, in, out);
  const int64_t ii = o % inner;
  const int64_t ro = o / inner;  // (row, outer) flattened
  const float* src = in + (ro * span + lo) * inner + ii;
  float acc = MAX ? -INFINITY : 0.0f;
  for (int64_t r = 0; r < red; ++r) {
    const float v = src[r * inner];
    acc = MAX ? fmaxf(acc, v) : acc + v;
  }
  out[o] = MAX ? acc : alpha * acc;
}

// inner a multiple of 4 (and aligned): one thread per four output elements, 128-bit streaming loads,
// four of them in flight per thread (the scalar form above keeps one 4-byte load per thread in
// flight and reaches 3 TB/s on the spin-wise means of a 16-electron layer; this one 5).
template <bool MAX>
__global__ __launch_bounds__(256) void reduce_mid_v4_kernel(Arrays arrays /* numbered by four outputs */, int64_t total4,
                                                            int64_t red, int64_t inner, int64_t span, int64_t lo,
                                                            float alpha) {
  int64_t o4 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (o4 >= total4) return;
  const float* in;
  float* out;
  arrays.find(o4, in, out);
  const int64_t inner4 = inner / 4;
  const int64_t ii = (o4 % inner4) * 4;
  const int64_t ro = o4 / inner4;  // (row, outer) flattened
  const float* src = in + (ro * span + lo) * inner + ii;
  const float init = MAX ? -INFINITY : 0.0f;
  float4 acc = make_float4(init, init, init, init);
  auto take = [&](const float4& v) {
    if (MAX) { acc.x = fmaxf(acc.x, v.x); acc.y = fmaxf(acc.y, v.y); acc.z = fmaxf(acc.z, v.z); acc.w = fmaxf(acc.w, v.w); }
    else { acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w; }
  };
  int64_t r = 0;
  for (; r + 4 <= red; r += 4) {  // in the order of the scalar kernel: r ascending
    const float4 v0 = folx_ld_stream4(src + (r + 0) * inner), v1 = folx_ld_stream4(src + (r + 1) * inner);
    const float4 v2 = folx_ld_stream4(src + (r + 2) * inner), v3 = folx_ld_stream4(src + (r + 3) * inner);
    take(v0); take(v1); take(v2); take(v3);
  }
  for (; r < red; ++r) take(folx_ld_stream4(src + r * inner));
  if (!MAX) { acc.x *= alpha; acc.y *= alpha; acc.z *= alpha; acc.w *= alpha; }
  *reinterpret_cast<float4*>(out + o4 * 4) = acc;
}

// inner == 1: G lanes (a power of two) per output element, each taking pieces of VEC consecutive values, U outputs of a
// group in flight.  Bound by HBM: G is the least that covers the reduced axis in one piece per lane, so that a wavefront
// reads one contiguous stretch (64 / G outputs side by side).  A whole wavefront per output left 48 of 64 lanes idle on
// the softmax sums of 16 particles: 1.6 M outputs of 16: 182 -> 17 us (6.6 TB/s); 5.7 M of 30: 826 -> 193 us.
// WAVE: G = 64 as a constant; a long axis read in single values is bound by its instructions (23 317 sums of 206: 7.6 -> 6.6 us,
// 29 035 of 434: 15.5 -> 14.4 us).
template <bool MAX, int VEC, int U, bool WAVE>
__global__ __launch_bounds__(256) void reduce_last_kernel(Arrays arrays, int64_t total, int64_t red, int64_t span,
                                                          int64_t lo, int32_t group, float alpha) {
  const int G = WAVE ? FOLX_WAVE : group;
  const int per = 256 / G, g = threadIdx.x / G, l = threadIdx.x % G;
  const int64_t o0 = (int64_t)blockIdx.x * (per * U) + g;
  const int64_t pieces = red / VEC;
  float acc[U];
  const float* src[U];
  float* dst[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    acc[u] = MAX ? -INFINITY : 0.0f;
    // outputs past the end read the last one's values
    int64_t o = o0 + u * per < total ? o0 + u * per : total - 1;
    const float* in;
    arrays.find(o, in, dst[u]);
    src[u] = in + o * span + lo;
    dst[u] += o;
  }
  for (int64_t r = l; r < pieces; r += G) {
    float v[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float* p = src[u] + r * VEC;
      if constexpr (VEC == 4) {
        const float4 q = folx_ld_stream4(p);
        v[u][0] = q.x; v[u][1] = q.y; v[u][2] = q.z; v[u][3] = q.w;
      } else {
        v[u][0] = *p;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[u] = MAX ? fmaxf(acc[u], v[u][i]) : acc[u] + v[u][i];
  }
  for (int off = G / 2; off > 0; off >>= 1)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float v = __shfl_xor(acc[u], off, FOLX_WAVE);
      acc[u] = MAX ? fmaxf(acc[u], v) : acc[u] + v;
    }
  if (l == 0)
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (o0 + u * per < total) *dst[u] = MAX ? acc[u] : alpha * acc[u];
}

template <bool MAX, int VEC>
int launch_reduce_last(hipStream_t st, const Arrays& a, int64_t total, int64_t red, int64_t span, int64_t lo, float alpha) {
  int G = 1;
  while (G < FOLX_WAVE && G < red / VEC) G *= 2;
  const int64_t per = 256 / G;
  // four outputs per group once that still leaves every CU several workgroups
  const int U = total >= 4 * per * 2048 ? 4 : 1;
  const int64_t blocks = (total + per * U - 1) / (per * U);
  if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
  const dim3 grid((unsigned)blocks), block(256);
  if (G == FOLX_WAVE) {
    if (U == 4) reduce_last_kernel<MAX, VEC, 4, true><<<grid, block, 0, st>>>(a, total, red, span, lo, G, alpha);
    else reduce_last_kernel<MAX, VEC, 1, true><<<grid, block, 0, st>>>(a, total, red, span, lo, G, alpha);
  } else {
    if (U == 4) reduce_last_kernel<MAX, VEC, 4, false><<<grid, block, 0, st>>>(a, total, red, span, lo, G, alpha);
    else reduce_last_kernel<MAX, VEC, 1, false><<<grid, block, 0, st>>>(a, total, red, span, lo, G, alpha);
  }
  return folx_launch_status();
}

// array k: outer[k] x (window of span) x inner
template <bool MAX>
int launch_reduce(hipStream_t st, int n, const float* const* in, float* const* out, const int64_t* outer, int64_t red,
                  int64_t inner, float alpha, int64_t span, int64_t lo) {
  if (red < 0 || inner < 0 || lo < 0 || lo + red > span) return FOLX_HIP_EINVAL;
  Arrays a;
  int64_t total = 0;
  bool in16 = true, out16 = true;
  int used = 0;
  for (int k = 0; k < n; ++k) {
    if (outer[k] < 0) return FOLX_HIP_EINVAL;
    if (outer[k] * inner == 0) continue;
    if (!in[k] || !out[k]) return FOLX_HIP_EINVAL;
    total += outer[k] * inner;
    a.in[used] = in[k]; a.out[used] = out[k]; a.end[used++] = total;
    in16 = in16 && folx_aligned16(in[k]);
    out16 = out16 && folx_aligned16(out[k]);
  }
  if (total == 0) return FOLX_HIP_OK;
  for (int k = used; k < 3; ++k) { a.in[k] = a.in[used - 1]; a.out[k] = a.out[used - 1]; a.end[k] = total; }
  if (inner == 1 && red >= 16) {
    if (red % 4 == 0 && span % 4 == 0 && lo % 4 == 0 && in16)
      return launch_reduce_last<MAX, 4>(st, a, total, red, span, lo, alpha);
    return launch_reduce_last<MAX, 1>(st, a, total, red, span, lo, alpha);
  } else if (inner % 4 == 0 && in16 && out16) {
    const int64_t blocks = (total / 4 + 255) / 256;
    if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
    for (int64_t& e : a.end) e /= 4;
    reduce_mid_v4_kernel<MAX><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(a, total / 4, red, inner, span, lo, alpha);
  } else {
    const int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7fffffffLL) return FOLX_HIP_ENOTSUP;
    reduce_mid_kernel<MAX><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(a, total, red, inner, span, lo, alpha);
  }
  return folx_launch_status();
}

template <bool MAX>
int launch_reduce(hipStream_t st, const float* in, float* out, int64_t rows, int64_t outer, int64_t red, int64_t inner,
                  float alpha, int64_t span, int64_t lo) {
  if (rows < 0 || outer < 0) return FOLX_HIP_EINVAL;
  const int64_t ro = rows * outer;
  return launch_reduce<MAX>(st, 1, &in, &out, &ro, red, inner, alpha, span, lo);
}

}  // namespace

extern "C" int folx_hip_reduce_sum(void* stream, const float* in, float* out, int64_t rows,
                                   int64_t outer, int64_t red, int64_t inner, float alpha) {
  return launch_reduce<false>((hipStream_t)stream, in, out, rows, outer, red, inner, alpha, red, 0);
}

extern "C" int folx_hip_reduce_sum_window(void* stream, const float* in, float* out, int64_t rows,
                                          int64_t outer, int64_t span, int64_t lo, int64_t hi, int64_t inner,
                                          float alpha) {
  if (hi < lo) return FOLX_HIP_EINVAL;
  return launch_reduce<false>((hipStream_t)stream, in, out, rows, outer, hi - lo, inner, alpha, span, lo);
}

extern "C" int folx_hip_reduce_max(void* stream, const float* in, float* out, int64_t outer,
                                   int64_t red, int64_t inner) {
  return launch_reduce<true>((hipStream_t)stream, in, out, 1, outer, red, inner, 1.0f, red, 0);
}

extern "C" int folx_hip_reduce_sum_arrays(void* stream, int32_t n, const float* const* in, float* const* out,
                                          const int64_t* outer, int64_t span, int64_t lo, int64_t hi, int64_t inner,
                                          float alpha) {
  if (n < 1 || n > 3 || !in || !out || !outer || hi < lo) return FOLX_HIP_EINVAL;
  return launch_reduce<false>((hipStream_t)stream, n, in, out, outer, hi - lo, inner, alpha, span, lo);
}
