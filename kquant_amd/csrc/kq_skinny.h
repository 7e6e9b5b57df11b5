// Linear for few activation rows: C[M, N] = A[M, K] x dequant(W)[N, K]^T on
// one weight pass, the K loop split over the waves of a workgroup.
//
// What bounds it: the weight bytes.  A 256 x 256 output tile pads a decode
// batch to 256 rows and leaves N / 256 workgroups on the chip, each streaming
// its weights alone; here a workgroup owns 16 R weight rows and every wave a
// contiguous run of 128-k windows of them, so N / (16 R) workgroups of
// independent waves keep the loads of the whole chip in flight.
//  * lane (r, g) of a wave (r = lane % 16, g = lane / 16) loads its weight row
//    with 16-byte loads: E4M3 windows as chunks 64 h + 16 g (h = 0, 1), E2M1
//    windows as the one chunk 32 g.  The 16x16x32 MFMA sums over any
//    assignment of k to (lane group, element), so the activations are read
//    with the same one and nothing is permuted.
//  * weights are expanded to bf16 in registers (exact); activations come
//    straight from memory (each wave has its own k, so LDS would hold
//    nothing twice): bf16 rows, fp32 rows split exactly into three bf16 terms
//    (one MFMA each), or MXFP8 rows, expanded like the weights: the products
//    are exact and sum in fp32, where the block-scaled fp8 MFMA drops bits of
//    a 128-product sum (3e-5 of the largest result at K = 128).
//  * P windows are in flight per wave; the last ones reload the wave's final
//    window instead of branching, so the compiler counts its waits exactly.
//  * the waves' partial tiles meet in LDS and are summed in wave order: no
//    atomics, no workspace, bitwise reproducible.
// Rows past M or N are read at the last valid row and not stored.
#pragma once

#include "kq_gemm.h"

namespace kq {
namespace skinny {

using gemm::bf16x8_t;
using gemm::u32x2_t;
using gemm::u32x4_t;
typedef float f32x4_t __attribute__((ext_vector_type(4)));

enum { A_BF16 = 0, A_F32 = 1, A_MXFP8 = 2 };
constexpr int WIN = 128;  // k per window

// One window of a wave: weight chunks and scale dwords of R row blocks,
// activation chunks of MB row blocks.
template <int FMT, int AT, int MB, int R>
struct Window {
  static constexpr int WC = FMT == 0 ? 2 : 1;
  static constexpr int AC = AT == A_F32 ? 8 : AT == A_MXFP8 ? 2 : 4;
  u32x4_t w[R][WC];
  uint32_t s[R];
  u32x4_t a[MB][AC];
  uint32_t as[MB];
};

__device__ __forceinline__ u32x4_t load16(const void* p) { return *static_cast<const u32x4_t*>(p); }
__device__ __forceinline__ u32x4_t load16_nt(const void* p) {
  return __builtin_nontemporal_load(static_cast<const u32x4_t*>(p));
}

// FMT: weight format; AT: activation rows; OUT: KQ_DT_BF16 / KQ_DT_F32;
// MB x 16 activation rows and R x 16 weight rows per workgroup, P windows in
// flight; HALF: K % 128 == 64 (2-byte aligned scale rows, a half window at
// the end).
template <int FMT, int AT, int OUT, int MB, int R, int P, bool HALF>
__global__ __launch_bounds__(512) void mx_skinny_kernel(
    const void* __restrict__ a, const uint8_t* __restrict__ a_scale, int64_t lda, const uint8_t* __restrict__ wq,
    const uint8_t* __restrict__ ws, void* __restrict__ c, int64_t ldc, int M, int N, int K, int mtiles) {
  static_assert(AT != A_MXFP8 || (FMT == 0 && !HALF), "MXFP8 rows take E4M3 weights and whole windows");
  using Win = Window<FMT, AT, MB, R>;
  extern __shared__ __attribute__((aligned(16))) float skinny_red[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int waves = (int)blockDim.x >> 6;
  // row tiles of one column tile run on one XCD, one after the other, and
  // share its weights in that L2
  const int idx = (int)blockIdx.x / 8, xcd = (int)blockIdx.x % 8;
  const int n0 = ((idx / mtiles) * 8 + xcd) * 16 * R, m0 = (idx % mtiles) * 16 * MB;
  if (n0 >= N) return;
  const int r = lane & 15, g = lane >> 4;
  const int nwin = (K + WIN - 1) / WIN;
  const int w_begin = (int)((int64_t)wave * nwin / waves), w_end = (int)((int64_t)(wave + 1) * nwin / waves);
  const int64_t kw = FMT == 0 ? K : K / 2, ks = K / 32;

  const uint8_t* wrow[R];
  const uint8_t* srow[R];
  const uint8_t* arow[MB];
  const uint8_t* asrow[MB];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int64_t n = min(n0 + 16 * j + r, N - 1);
    wrow[j] = wq + n * kw + 16 * g;
    srow[j] = ws + n * ks;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int64_t m = min(m0 + 16 * i + r, M - 1);
    const int esize = AT == A_F32 ? 4 : AT == A_BF16 ? 2 : 1;
    arow[i] = static_cast<const uint8_t*>(a) + (m * lda + (FMT == 0 ? 16 : 32) * g) * esize;
    asrow[i] = AT == A_MXFP8 ? a_scale + m * ks : nullptr;
  }

  auto load = [&](int w, Win& v) {
    const int64_t k0 = (int64_t)w * WIN;
    const bool half = HALF && k0 + WIN > K;  // only the last window of a K % 128 == 64 row
    // E4M3: the second chunk of a half window is past the row; E2M1: the chunks of g = 2, 3 are
    const bool cut = half && (FMT == 0 || g >= 2);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (FMT == 0) {
        v.w[j][0] = load16_nt(wrow[j] + k0);
        v.w[j][Win::WC - 1] = load16_nt(wrow[j] + k0 + (cut ? 0 : 64));
        if (cut) v.w[j][Win::WC - 1] = u32x4_t{0u, 0u, 0u, 0u};
      } else {
        v.w[j][0] = load16_nt(wrow[j] + k0 / 2 - (cut ? 32 : 0));
        if (cut) v.w[j][0] = u32x4_t{0u, 0u, 0u, 0u};
      }
      if (HALF) {
        const uint16_t* sp = reinterpret_cast<const uint16_t*>(srow[j] + k0 / 32);
        v.s[j] = (uint32_t)sp[0] | (uint32_t)sp[half ? 0 : 1] << 16;
      } else {
        v.s[j] = *reinterpret_cast<const uint32_t*>(srow[j] + k0 / 32);
      }
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      if (AT == A_MXFP8) {
        v.a[i][0] = load16(arow[i] + k0);
        v.a[i][1] = load16(arow[i] + k0 + 64);
        v.as[i] = *reinterpret_cast<const uint32_t*>(asrow[i] + k0 / 32);
      } else {
        constexpr int ES = AT == A_F32 ? 4 : 2, PER = AT == A_F32 ? 2 : 1;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int koff = FMT == 0 ? 64 * (t >> 1) + 8 * (t & 1) : 8 * t;
          const bool gone = cut && (FMT == 1 || t >= 2);
          const uint8_t* p = arow[i] + (k0 + (gone ? koff - 64 : koff)) * ES;
#pragma unroll
          for (int e = 0; e < PER; ++e) {
            v.a[i][PER * t + e] = load16(p + 16 * e);
            if (gone) v.a[i][PER * t + e] = u32x4_t{0u, 0u, 0u, 0u};
          }
        }
      }
    }
  };

  f32x4_t acc[MB][R];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // MXFP8 rows: E4M3 x 2^(s - 127) is a normal bf16 for 10 <= s <= 246; a
  // window with another scale byte (any lane's) is left for after the loop
  auto odd_scales = [&](const Win& v) -> bool {
    bool odd = false;
#pragma unroll
    for (int j = 0; j < R; ++j) odd |= (v.s[j] >> (8 * g) & 0xffu) - 10u > 236u;
#pragma unroll
    for (int i = 0; i < MB; ++i) odd |= (v.as[i] >> (8 * g) & 0xffu) - 10u > 236u;
    return __any(odd);
  };
  bool left = false;

  auto compute = [&](const Win& v) {
    if constexpr (AT == A_MXFP8) {
      if (odd_scales(v)) {
        left = true;
        return;
      }
    }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        bf16x8_t fa[MB][AT == A_F32 ? 3 : 1];
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          if constexpr (AT == A_F32) {
            // v = a0 + a1 + a2 exactly: 8 significant bits each, every residual exact
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float x = __uint_as_float(v.a[i][2 * t + (e >> 2)][e & 3]);
              const __bf16 h0 = (__bf16)x;
              const float r1 = x - (float)h0;
              const __bf16 h1 = (__bf16)r1;
              fa[i][0][e] = h0;
              fa[i][1][e] = h1;
              fa[i][2][e] = (__bf16)(r1 - (float)h1);
            }
          } else if constexpr (AT == A_MXFP8) {
            fa[i][0] = gemm::dequant8<0>(u32x2_t{v.a[i][t >> 1][2 * (t & 1)], v.a[i][t >> 1][2 * (t & 1) + 1]},
                                         v.as[i] >> (16 * (t >> 1) + 8 * (g >> 1)) & 0xffu);
          } else {
            fa[i][0] = __builtin_bit_cast(bf16x8_t, v.a[i][t]);
          }
        }
#pragma unroll
        for (int j = 0; j < R; ++j) {
          u32x2_t w;
          uint32_t sb;
          if (FMT == 0) {
            w = u32x2_t{v.w[j][t >> 1][2 * (t & 1)], v.w[j][t >> 1][2 * (t & 1) + 1]};
            sb = v.s[j] >> (16 * (t >> 1) + 8 * (g >> 1)) & 0xffu;
          } else {
            w = u32x2_t{v.w[j][0][t], 0u};
            sb = v.s[j] >> (8 * g) & 0xffu;
          }
          const bf16x8_t fb = gemm::dequant8<FMT>(w, sb);
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int x = 0; x < (AT == A_F32 ? 3 : 1); ++x)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i][x], fb, acc[i][j], 0, 0, 0);
        }
      }
  };

  if (w_begin < w_end) {
    Win v[P];
#pragma unroll
    for (int p = 0; p < P; ++p) load(min(w_begin + p, w_end - 1), v[p]);
    int w = w_begin;
    for (; w + P <= w_end; w += P) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        compute(v[p]);
        load(min(w + P + p, w_end - 1), v[p]);
      }
    }
#pragma unroll
    for (int p = 0; p < P - 1; ++p)
      if (w + p < w_end) compute(v[p]);
  }

  if constexpr (AT == A_MXFP8) {
    // The windows left: the codes themselves multiply in fp32, each 32-k block
    // on its own (lane groups 2 blk and 2 blk + 1 of its chunk; element e of
    // every lane is one k of a 16x16x4 MFMA), and both scales apply to the
    // block's sum as one exponent, so an operand may leave fp32's range where
    // the product does not.  Scale byte 255 is NaN.
    for (int w = w_begin; left && w < w_end; ++w) {
      Win v;
      load(w, v);
      if (!odd_scales(v)) continue;
#pragma nounroll
      for (int blk = 0; blk < 4; ++blk) {
        const bool mine = (g >> 1) == (blk & 1);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j) {
            f32x4_t dot = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
              const uint32_t aw = blk & 2 ? v.a[i][1][e >> 2] : v.a[i][0][e >> 2];
              const uint32_t ww = !mine ? 0u : blk & 2 ? v.w[j][1][e >> 2] : v.w[j][0][e >> 2];
              const float2_t x = e & 2 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(aw, 1.0f, true)
                                       : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(aw, 1.0f, false);
              const float2_t b = e & 2 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(ww, 1.0f, true)
                                       : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(ww, 1.0f, false);
              dot = __builtin_amdgcn_mfma_f32_16x16x4f32(x[0], b[0], dot, 0, 0, 0);
              dot = __builtin_amdgcn_mfma_f32_16x16x4f32(x[1], b[1], dot, 0, 0, 0);
            }
            const int sw = (int)(v.s[j] >> (8 * blk) & 0xffu);
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // row 4 g + q: lane 4 g + q has its scales
              const int sa = (int)((uint32_t)__shfl((int)v.as[i], 4 * g + q) >> (8 * blk) & 0xffu);
              const float term = __builtin_amdgcn_ldexpf(dot[q], sa + sw - 254);
              acc[i][j][q] += sa == 255 || sw == 255 ? __builtin_nanf("") : term;
            }
          }
      }
    }
  }

  // D (16x16): lane holds column lane % 16, rows 4 (lane / 16) + j
  constexpr int TILE = MB * R * 256;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j)
      *reinterpret_cast<f32x4_t*>(skinny_red + wave * TILE + (i * R + j) * 256 + lane * 4) = acc[i][j];
  __syncthreads();
  for (int e = (int)threadIdx.x; e < TILE; e += (int)blockDim.x) {
    const int n = e % (16 * R), m = e / (16 * R);
    if (m0 + m >= M || n0 + n >= N) continue;
    const int at = ((m >> 4) * R + (n >> 4)) * 256 + (16 * ((m & 15) >> 2) + (n & 15)) * 4 + (m & 3);
    float sum = skinny_red[at];
    for (int w = 1; w < waves; ++w) sum += skinny_red[w * TILE + at];
    if (OUT == 2) static_cast<float*>(c)[(int64_t)(m0 + m) * ldc + n0 + n] = sum;
    else static_cast<__bf16*>(c)[(int64_t)(m0 + m) * ldc + n0 + n] = (__bf16)sum;
  }
}

}  // namespace skinny
}  // namespace kq
