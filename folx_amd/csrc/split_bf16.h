// FP32 products on the bf16 matrix pipe: every operand is split into three bf16 pieces,
//     x = x1 + x2 + x3   (x1 = bf16(x), x2 = bf16(x - x1), x3 = bf16(x - x1 - x2), exact: 3 x 8
//                         significand bits cover the 24 of an fp32 number),
// and a product a b is taken as the six piece products of weight >= 2^-16,
//     a3 b1 + a2 b2 + a2 b1 + a1 b3 + a1 b2 + a1 b1,
// each exact in fp32 and summed in the fp32 accumulator of v_mfma_f32_32x32x16_bf16.  The three
// products that are left out (a2 b3, a3 b2, a3 b3) weigh <= 2^-24 of a b, the rounding of one
// fp32 multiply-add.  Six bf16 products of depth 16 take 6 x 8 passes on the matrix pipe for
// the work of 8 v_mfma_f32_32x32x2_f32 (8 x 16 passes): 2.7 times the FP32 rate.
//
// An infinite element (or one that rounds to a bf16 infinity) turns into NaN: x - bf16(x) is
// inf - inf.  Finite inputs, the case the rules are used for, are represented exactly.
//
// The mode is process wide (folx_hip_set_gemm_mode); kernels that have no split form ignore it.
#pragma once
#include "common.h"

// 0: v_mfma_f32_32x32x2_f32 on the fp32 operands; 1: the split above where a kernel has it
int folx_gemm_mode();

#ifdef __HIPCC__
#include <type_traits>

namespace folx_split {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

// Two numbers at once (v_cvt_pk_bf16_f32 rounds a pair to nearest even): piece i of x in the
// low half of pi, of y in the high half.
__device__ __forceinline__ void split_pair(float x, float y, unsigned& p1, unsigned& p2, unsigned& p3) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  auto cvt = [](float a, float b) -> unsigned {
    f2 v;
    v[0] = a;
    v[1] = b;
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf2));
  };
  p1 = cvt(x, y);
  float rx = x - __uint_as_float(p1 << 16), ry = y - __uint_as_float(p1 & 0xffff0000u);
  p2 = cvt(rx, ry);
  rx -= __uint_as_float(p2 << 16);
  ry -= __uint_as_float(p2 & 0xffff0000u);
  p3 = cvt(rx, ry);
}

// The six products in the order they are accumulated: by A piece (one piece of A in
// registers at a time), small terms before the leading one.
constexpr int kPieceA[6] = {2, 1, 1, 0, 0, 0};
constexpr int kPieceB[6] = {0, 1, 0, 2, 1, 0};


// The pieces of a weight matrix W (K x N, K a multiple of 16), prepared once per call and laid out as the tiles below take them:
//   [K / 16][piece][column / 32][k / 8 within the chunk][column % 32][8 bf16]
// (columns padded to a multiple of 32 with zeros), so that 32 columns of a chunk and piece are 1 KB in a row.
inline int64_t pieces_bytes(int32_t K, int32_t N) { return (int64_t)K * ((N + 31) / 32 * 32) * 6; }

// Infinite and NaN weights keep their first piece only (the others would be NaN), and a finite one that rounds to a bf16
// infinity is cut instead of rounded: w1 + w2 + w3 is the weight for every float.
__device__ __forceinline__ void split_weight(float x, unsigned short& p1, unsigned short& p2, unsigned short& p3) {
  unsigned a, b, c;
  split_pair(x, x, a, b, c);
  if ((a & 0x7f80u) == 0x7f80u) {
    const unsigned u = __float_as_uint(x);
    a = u >> 16;
    b = c = 0;
    if ((u & 0x7f800000u) == 0x7f800000u) {
      if (x != x) a |= 0x40u;
    } else {
      unsigned d;
      split_pair(x - __uint_as_float(u & 0xffff0000u), 0.0f, b, c, d);
    }
  }
  p1 = (unsigned short)a; p2 = (unsigned short)b; p3 = (unsigned short)c;
}

// Eight consecutive k (an octet) of column n
__device__ __forceinline__ void store_octet(const float (&w)[8], char* out, int32_t octet, int32_t n, int32_t blocks) {
  typedef unsigned short ushort8 __attribute__((ext_vector_type(8)));
  ushort8 p[3];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    unsigned short a, b, c;
    split_weight(w[e], a, b, c);
    p[0][e] = a; p[1][e] = b; p[2][e] = c;
  }
  char* to = out + ((int64_t)(octet / 2) * 3 * blocks + n / 32) * 1024 + (octet % 2) * 512 + (n % 32) * 16;
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<ushort8*>(to + (int64_t)q * blocks * 1024) = p[q];
}

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx16 zeros() {
  floatx16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.0f;
  return z;
}

#define FOLX_SPLIT_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define FOLX_SPLIT_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

// The products of one tile: a workgroup of 4 wavefronts takes 128 rows x 32 CB columns, wavefront w rows 32 w .. 32 w + 31 of
// ALL columns.  Nobody else multiplies a wavefront's rows, so A never goes through LDS: a lane asks for the 8 k of its row that
// the matrix instruction wants from it (row lane % 32, k = 16 chunk + 8 (lane / 32) + 0 .. 7), two chunks ahead, and splits
// them in registers.  The pieces of W go from memory (L2) straight into LDS, one chunk ahead; a fragment read is 1 KB in a row.
// One barrier a chunk.
//
// What bounds it: the power cap.  us, K = N = 256, 3.2 M rows, fp32 instructions -> here: plain 3350 -> 2330, with a skip connection
// 3650 -> 2680, behind LayerNorm 3670 -> 2700, behind LayerNorm with tanh 3760 -> 2780 (W and A both through registers into LDS, 8
// wavefronts of 64 x 64: 2420, 2730, 2840, 2910), at a clock of 1.6 GHz; the products alone, without the traffic of A and C, 1750
// (three products instead of six: 1000; one: 600).  What counts is energy: splitting W in every workgroup instead of once
// costs 250 us (88 vector instructions beside 48 matrix ones a chunk and wavefront).  The scheduler has to be kept from moving the
// fragment reads of the next block of columns behind the products of this one: 100 us.
//
// An element that is infinite, NaN or rounds to a bf16 infinity shows as a sum that is not finite; a wavefront that
// has one takes its products again with the fp32 instructions, from the original A and the sum of W's pieces, for the sums concerned.
// ONE_LOOP: full tiles and those with fewer blocks run the same loop (accumulators that do not start from constants would be
// copied in front of each of two loops, and spilled).
// APART: the products of a chunk are summed apart and added to the running sum once, which rounds against it once in 16 k instead
// of six times, for 16 additions more beside six products.  For sums of more than APART_K products.
constexpr int APART_K = 512;
// FLY: W is split by every workgroup on its way into LDS instead of once per call, thread t 16 CB / 8 consecutive k of column
// t % (32 CB): for launches of few workgroups, where one launch more would cost as much as the products.
// LDS traffic of this workgroup is complete; requests on their way to memory stay on their way
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// KEEP: and writes the pieces to memory as well.
template <int CB, bool ONE_LOOP = false, bool APART = false, bool FLY = false, bool KEEP = false>
struct SplitTile {
  static constexpr int NT = 256, BM = 128, BN = 32 * CB;
  static constexpr int KPT = 16 * BN / NT;  // FLY: k of a chunk that a thread stages
  static constexpr int D = 2;  // chunks asked for ahead (4 with FLY: no faster, 24 registers more)
  static constexpr int PLANE = CB * 1024;  // bytes of one piece of a W chunk
  static constexpr int STAGE = 3 * PLANE;

  // acc[0][j] = start(j) + rows x columns 32 j .. 32 j + 31, j < nb; init() sets acc to all of start.  w: the pieces of the tile's first block, of `blocks` in a
  // chunk and piece (FLY: where this workgroup writes them, or NULL, and W the weights from the tile's first column, `cols` to
  // the right of it and rows of N); at(kt): the lane's 8 floats of chunk kt (16-byte aligned); seen(kt, v0, v1): the same floats, once each;
  // meanwhile(): work while the first chunk is on its way, what it writes to LDS is there for seen() and after the call.
  template <class Start, class Init, class At, class Seen, class Meanwhile>
  static __device__ __forceinline__ void products(floatx16 (&acc)[1][CB], char* ws0, char* ws1, const char* __restrict__ w,
                                                  int32_t blocks, int32_t nb, int32_t KT, Start start, Init init, At at, Seen seen,
                                                  Meanwhile meanwhile, const float* __restrict__ W = nullptr, int32_t N = 0,
                                                  int32_t cols = 0) {
    const int lane = threadIdx.x % 64, wave = folx_wave_id();
    const int64_t plane = (int64_t)blocks * 1024;
    // FLY: this thread's column and first k, where its pieces go in a plane, and the k of the next chunk in registers
    const int wcol = threadIdx.x % BN, wk = threadIdx.x / BN * KPT;
    const float* w_src = W + (int64_t)wk * N + (wcol < cols ? wcol : cols - 1);
    const int w_dst = (wcol / 32) * 1024 + (wk / 8) * 512 + (wcol % 32) * 16 + (wk % 8) * 2;
    float rws[FLY ? D : 1][FLY ? KPT : 1];
    auto load_w = [&](int kt, auto& rw) __attribute__((always_inline)) {
      const float* p = w_src + (int64_t)(kt < KT ? kt : KT - 1) * 16 * N;
#pragma unroll
      for (int e = 0; e < KPT; ++e) rw[e] = p[(int64_t)e * N];
    };
    auto put = [&](const unsigned (&p)[3][KPT / 2], char* to, int64_t step) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        if constexpr (KPT == 8) *reinterpret_cast<uint4v*>(to + q * step) = uint4v{p[q][0], p[q][1], p[q][2], p[q][3]};
        else *reinterpret_cast<uint2v*>(to + q * step) = uint2v{p[q][0], p[q][1]};
      }
    };
    auto put_w = [&](char* ws, auto& rw) __attribute__((always_inline)) {
      unsigned p[3][KPT / 2];
#pragma unroll
      for (int c = 0; c < KPT / 2; ++c) split_pair(rw[2 * c], rw[2 * c + 1], p[0][c], p[1][c], p[2][c]);
      put(p, ws + w_dst, PLANE);
    };
    auto keep_w = [&](int kt, auto& rw) __attribute__((always_inline)) {  // the pieces for whoever comes after this launch
      unsigned p[3][KPT / 2];
#pragma unroll
      for (int c = 0; c < KPT / 2; ++c) {
        unsigned short u[3], v[3];
        split_weight(wcol < cols ? rw[2 * c] : 0.0f, u[0], u[1], u[2]);
        split_weight(wcol < cols ? rw[2 * c + 1] : 0.0f, v[0], v[1], v[2]);
#pragma unroll
        for (int q = 0; q < 3; ++q) p[q][c] = u[q] | (unsigned)v[q] << 16;
      }
      if (w != nullptr && wcol / 32 < nb) put(p, const_cast<char*>(w) + (int64_t)kt * 3 * plane + w_dst, plane);
    };
    float4 ra[D][2];
    bf16x8 fa[3];
    auto fetch_a = [&](int kt, float4 (&r)[2]) __attribute__((always_inline)) {
      if (!FLY && kt >= KT) return;
      const float4v* p = reinterpret_cast<const float4v*>(at(FLY && kt >= KT ? KT - 1 : kt));
      const auto* g = (const __attribute__((address_space(1))) float4v*)p;
      const float4v u = g[0], v = g[1];  // plain: the line's other half follows one chunk later
      r[0] = make_float4(u[0], u[1], u[2], u[3]);
      r[1] = make_float4(v[0], v[1], v[2], v[3]);
    };
    auto fetch_w = [&](int kt, char* ws, auto all) __attribute__((always_inline)) {
      if (kt >= KT) return;
      const char* p = w + (int64_t)kt * 3 * plane + lane * 16;
#pragma unroll
      for (int i = 0; i < (3 * CB + 3) / 4; ++i) {
        const int u = wave + 4 * i;  // 1 KB of the stage
        if (3 * CB % 4 != 0 && u >= 3 * CB) continue;
        if (decltype(all)::value || u % CB < nb)
          __builtin_amdgcn_global_load_lds(FOLX_SPLIT_GPTR(p + (u / CB) * plane + (u % CB) * 1024), FOLX_SPLIT_LPTR(ws + u * 1024),
                                           16, 0, 0);
      }
    };
    auto split_a = [&](const float4 (&r)[2]) __attribute__((always_inline)) {
      unsigned p1[4], p2[4], p3[4];
      split_pair(r[0].x, r[0].y, p1[0], p2[0], p3[0]);
      split_pair(r[0].z, r[0].w, p1[1], p2[1], p3[1]);
      split_pair(r[1].x, r[1].y, p1[2], p2[2], p3[2]);
      split_pair(r[1].z, r[1].w, p1[3], p2[3], p3[3]);
      fa[0] = __builtin_bit_cast(bf16x8, uint4v{p1[0], p1[1], p1[2], p1[3]});
      fa[1] = __builtin_bit_cast(bf16x8, uint4v{p2[0], p2[1], p2[2], p2[3]});
      fa[2] = __builtin_bit_cast(bf16x8, uint4v{p3[0], p3[1], p3[2], p3[3]});
    };

    if constexpr (FLY) {
#pragma unroll
      for (int u = 0; u < D; ++u) load_w(u, rws[u]);
    } else {
      fetch_w(0, ws0, std::false_type{});
    }
#pragma unroll
    for (int u = 0; u < D; ++u) fetch_a(u, ra[u]);
    meanwhile();
    init();
    if constexpr (FLY) {
      put_w(ws0, rws[0]);
      if constexpr (KEEP) keep_w(0, rws[0]);
      load_w(D, rws[0]);
      split_a(ra[0]);
      fetch_a(D, ra[0]);
      lds_barrier();
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }

    // FLY: chunk kt from stage ws and the pieces of A in registers; r, rw: chunk kt + 1 of A and W.  One block of code without branches, so
    // that the scheduler puts the splitting of the next chunk between the products of this one: few wavefronts share a SIMD here,
    // and a product waits for the one before it on the same block.
    auto chunk_fly = [&](int kt, const char* ws, char* next, float4 (&r)[2], auto& rw) __attribute__((always_inline)) {
      const char* f = ws + lane * 16;
      bf16x8 fb[CB][3];
#pragma unroll
      for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int p = 0; p < 3; ++p) fb[j][p] = *reinterpret_cast<const bf16x8*>(f + p * PLANE + j * 1024);
      __builtin_amdgcn_sched_barrier(0);  // all at once, not each in front of its use
      floatx16 sum[CB];
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if constexpr (APART) {
#pragma unroll
          for (int i = 0; i < 16; ++i) sum[j][i] = 0.0f;
        } else {
          sum[j] = acc[0][j];
        }
      }
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < CB; ++j)
          sum[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kPieceA[q]], fb[j][kPieceB[q]], sum[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if constexpr (APART) acc[0][j] += sum[j];
        else acc[0][j] = sum[j];
      }
      put_w(next, rw);
      seen(kt + 1, r[0], r[1]);
      split_a(r);
      fetch_a(kt + 1 + D, r);
      if constexpr (KEEP)
        if (kt + 1 < KT) keep_w(kt + 1, rw);
      load_w(kt + 1 + D, rw);
      lds_barrier();
    };
    // chunk kt from stage ws; chunk kt + 1 of W goes to the other stage, kt + 2 of A is asked for
    auto chunk = [&](int kt, const char* ws, char* next, float4 (&r)[2], auto all) __attribute__((always_inline)) {
      constexpr bool ALL = decltype(all)::value;
      const char* f = ws + lane * 16;
      bf16x8 fb[2][3];  // one block's fragments, the next one's on their way
      auto read = [&](int j, bf16x8 (&b)[3]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 3; ++p) b[p] = *reinterpret_cast<const bf16x8*>(f + p * PLANE + j * 1024);
      };
      read(0, fb[0]);
      seen(kt, r[0], r[1]);
      split_a(r);
      __builtin_amdgcn_sched_barrier(0);  // (the compiler waits for everything in front of r)
      fetch_w(kt + 1, next, all);
      fetch_a(kt + 2, r);
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if (j + 1 < CB) read(j + 1, fb[(j + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        if (ALL || j < nb) {
          floatx16 sum;
          if constexpr (APART) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = 0.0f;
          } else {
            sum = acc[0][j];
          }
#pragma unroll
          for (int q = 0; q < 6; ++q)
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kPieceA[q]], fb[j & 1][kPieceB[q]], sum, 0, 0, 0);
          if constexpr (APART) acc[0][j] += sum;
          else acc[0][j] = sum;
        }
      }
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    auto loop = [&](auto all) __attribute__((always_inline)) {
      for (int kt = 0; kt < KT; kt += 2) {
        chunk(kt, ws0, ws1, ra[0], all);
        if (kt + 1 < KT) chunk(kt + 1, ws1, ws0, ra[1], all);
      }
    };
    if constexpr (FLY) {
      for (int kt = 0; kt < KT; kt += D) {
#pragma unroll
        for (int u = 0; u < D; ++u)
          if (kt + u < KT) chunk_fly(kt + u, u % 2 ? ws1 : ws0, u % 2 ? ws0 : ws1, ra[(u + 1) % D], rws[(u + 1) % D]);
      }
    } else if constexpr (ONE_LOOP) {
      loop(std::false_type{});
    } else {
      if (nb >= CB) loop(std::true_type{});
      else loop(std::false_type{});
    }

    // A bad element of A spoils its whole row, one of W its whole column: one column and one row tell.
    float finite = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) finite = fmaf(acc[0][0][r], 0.0f, finite);
#pragma unroll
    for (int j = 1; j < CB; ++j) finite = fmaf(acc[0][j][0], 0.0f, finite);
    if (__any(!(finite == 0.0f))) {
      const int l32 = lane % 32, lh = lane / 32;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if (j >= nb) continue;
        floatx16 sum = start(j);
#pragma unroll 1
        for (int kt = 0; kt < KT; ++kt) {
          const auto* arow = (const __attribute__((address_space(1))) float*)(at(kt) - 8 * lh);
#pragma unroll 1
          for (int s = 0; s < 8; ++s) {
            const int k = 2 * s + lh;
            float wv;
            if constexpr (FLY) {
              const int n = 32 * j + l32;
              wv = W[(int64_t)(16 * kt + k) * N + (n < cols ? n : cols - 1)];
            } else {
              const char* wp = w + (int64_t)kt * 3 * plane + (k / 8) * 512 + l32 * 16 + (k % 8) * 2;
              auto piece = [&](int q) __attribute__((always_inline)) {
                return __uint_as_float((unsigned)*reinterpret_cast<const unsigned short*>(wp + q * plane + j * 1024) << 16);
              };
              wv = (piece(0) + piece(1)) + piece(2);
            }
            sum = __builtin_amdgcn_mfma_f32_32x32x2f32(arow[k], wv, sum, 0, 0, 0);
          }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r)  // the other sums stay what they are without such a neighbour
          acc[0][j][r] = fabsf(acc[0][j][r]) < __builtin_inff() ? acc[0][j][r] : sum[r];
      }
    }
  }
};

}  // namespace folx_split
#endif
