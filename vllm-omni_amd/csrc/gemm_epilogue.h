// The elementwise tail of the hand-written GEMM kernels: what happens to 8 consecutive output features of
// one row on their way from the fp32 accumulators to memory (bias, GELU(tanh), gate, residual, rounding).
// Shared by the stream-K kernel for few rows (gemm_bf16.hip) and the tile kernel for many (gemm_tile.h).
#pragma once

#include <type_traits>

#include "attn_common.h"
#include "gemm_bf16.h"

namespace odit {

template <typename T> struct Mma16;
template <> struct Mma16<bf16_t> {
  using frag = bf16x8_v;
  static __device__ __forceinline__ f32x4_v run(frag a, frag b, f32x4_v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma16<f16_t> {
  using frag = f16x8_v;
  static __device__ __forceinline__ f32x4_v run(frag a, frag b, f32x4_v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

struct GemmEpilogue {
  const void *bias, *residual, *gate;
  void* out;
  int M, N;
  int64_t ldo, ldr, ldg;
  int epilogue, gate_f32, rows_per_gate;
  float most;  // largest size of a gated result of f16 (infinite: as it comes)
};

// Held to a size of at most `most`; a NaN stays one.
__device__ __forceinline__ float f16_clipped(float y, float most = 65504.f) { return __builtin_elementwise_minimum(__builtin_elementwise_maximum(y, -most), most); }

// A gated result as ODIT_LINEAR_CLIP asks for it. Clipped before it is rounded: what rounds to infinity lies above the largest finite value, so
// these are the bits of a clip behind the rounding. That was a pass of its own over each stream behind every block; whole models in f16, width
// 3072, with it and without (us): 1085 + 44 rows, four blocks, 2511 and 2466; 169 + 121 and 269, five, 1852 and 1811; 6156 + 44, six, 19796 and 19714.
template <typename T> __device__ __forceinline__ float gemm_clipped(const GemmEpilogue& e, float y) {
  if constexpr (std::is_same<T, f16_t>::value) return f16_clipped(y, e.most);
  else return y;
}

// x sigmoid(2 u) of gemm_gelu_tanh, with the hardware's power and reciprocal as they come and 1 - 1 / (1 + e^(2 u)) for the sigmoid: the operations that
// give the library's results (bf16, none of 33 million differs; 0.4 % of those are not the nearest to float64's).
// Minus infinity gives NaN, as there; arguments of more than half the largest number themselves, where the library overflows.
__device__ __forceinline__ float gemm_gelu_apart(float x) {
#pragma clang fp contract(off)
  const float e = __builtin_amdgcn_exp2f(x * fmaf(x * 0.044715f, x, 1.f) * static_cast<float>(0.7978845608028654 * 2.885390081777927));
  return x * (1.f - __builtin_amdgcn_rcpf(e + 1.f));
}

// gate * sum + residual + bias with a rounding each, in the order in which the library's epilogue does it: its bits (4.2 million results of exact sums; one fma
// less in the other order, or one more, differs in 10 to 40 of a million)
__device__ __forceinline__ float gemm_gated_apart(float a, float gate, float residual, float bias) {
#pragma clang fp contract(off)
  return (a * gate + residual) + bias;
}

__device__ __forceinline__ float gemm_gelu_tanh(float x) {
  // x sigmoid(2 u), u = sqrt(2/pi) (x + 0.044715 x^3), with e^(-2 u) as a power of two. 48 elements per lane wait here with
  // nothing to overlap, so the quotient is the hardware reciprocal (1 ulp) with one correction by the remainder, six
  // instructions where the compiler's division takes ten. Error against float64 (2-norm, relative; reciprocal alone / corrected /
  // x / (1 + exp) in float32): N(0,1) 4.71e-8 / 4.21e-8 / 4.32e-8, N(0,0.01) 5.18e-8 / 4.37e-8 / 4.37e-8, N(0,3) 3.50e-8 /
  // 3.34e-8 / 3.35e-8. Time at N=12288, K=3072 (M = 80 / 256 / 512 / 1024), reciprocal alone 30.3 / 36.4 / 47.3 / 90.4 us,
  // corrected 31.1 / 37.2 / 48.0 / 91.9.
  const float e = __builtin_amdgcn_exp2f(x * fmaf(x * x, -2.f * 0.7978845608028654f * 0.044715f * 1.4426950408889634f,
                                                  -2.f * 0.7978845608028654f * 1.4426950408889634f));
  const float d = 1.f + e, r = __builtin_amdgcn_rcpf(d), q = x * r, rem = fmaf(-q, d, x);
  // (a zero remainder: q is exact; an infinite or NaN one: x or d is infinite and q is the limit)
  return __builtin_amdgcn_classf(rem, 0x198) ? fmaf(rem, r, q) : q;
}

// Features n .. n + 7 (n a multiple of 8, n < N) of what row m's accumulators y are combined with: y * gt + bs (+ the residual)
// for the gated epilogues, y + bs for the others.
template <typename T>
__device__ __forceinline__ void gemm_epilogue_vectors8(const GemmEpilogue& p, int m, int n, float (&gt)[8], float (&bs)[8]) {
  const T* bias_h = static_cast<const T*>(p.bias);
  const float* bias_f = static_cast<const float*>(p.bias);
  const bool gated = p.epilogue == ODIT_EPI_GATED_RESIDUAL || p.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
  const bool pre = p.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
#pragma unroll
  for (int u = 0; u < 8; ++u) { gt[u] = 1.f; bs[u] = 0.f; }
  const int64_t grow = gated && p.rows_per_gate > 0 ? static_cast<int64_t>(m / p.rows_per_gate) * p.ldg : 0;
  if (gated && p.gate != nullptr) {
    if (p.gate_f32) {
      const float* gp = static_cast<const float*>(p.gate) + grow + n;
      const f32x4_v g0 = *reinterpret_cast<const f32x4_v*>(gp), g1 = *reinterpret_cast<const f32x4_v*>(gp + 4);
#pragma unroll
      for (int u = 0; u < 4; ++u) { gt[u] = g0[u]; gt[4 + u] = g1[u]; }
    } else {
      const u32x4 gv = load_raw(static_cast<const T*>(p.gate) + grow + n);
#pragma unroll
      for (int u = 0; u < 8; ++u) gt[u] = Raw<T>::get(gv, u);
    }
  }
  if (p.bias != nullptr) {
    if (pre) {  // float32, already multiplied by the gate, one vector per gate vector
      const float* bp = bias_f + grow + n;
      const f32x4_v b0 = *reinterpret_cast<const f32x4_v*>(bp), b1 = *reinterpret_cast<const f32x4_v*>(bp + 4);
#pragma unroll
      for (int u = 0; u < 4; ++u) { bs[u] = b0[u]; bs[4 + u] = b1[u]; }
    } else {
      const u32x4 bv = load_raw(bias_h + n);
#pragma unroll
      for (int u = 0; u < 8; ++u) bs[u] = gated ? gt[u] * Raw<T>::get(bv, u) : Raw<T>::get(bv, u);
    }
  }
}

// y[0..8) = accumulators of row m, features n .. n + 7 (n a multiple of 8, m < M, n < N): applies the
// epilogue and stores 16 bytes
template <typename T>
__device__ __forceinline__ void gemm_epilogue_store8(const GemmEpilogue& p, int m, int n, float (&y)[8]) {
  const T* bias_h = static_cast<const T*>(p.bias);
  const float* bias_f = static_cast<const float*>(p.bias);
  const bool gelu = p.epilogue == ODIT_EPI_GELU_TANH || p.epilogue == ODIT_EPI_BIAS_GELU_TANH;
  const bool gated = p.epilogue == ODIT_EPI_GATED_RESIDUAL || p.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
  const bool pre = p.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
  if (gated) {
    const int64_t grow = p.rows_per_gate > 0 ? static_cast<int64_t>(m / p.rows_per_gate) * p.ldg : 0;
    float gt[8], bs[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) { gt[u] = 1.f; bs[u] = 0.f; }
    if (p.gate != nullptr) {
      if (p.gate_f32) {
        const float* gp = static_cast<const float*>(p.gate) + grow + n;
        const f32x4_v g0 = *reinterpret_cast<const f32x4_v*>(gp), g1 = *reinterpret_cast<const f32x4_v*>(gp + 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) { gt[u] = g0[u]; gt[4 + u] = g1[u]; }
      } else {
        const u32x4 gv = load_raw(static_cast<const T*>(p.gate) + grow + n);
#pragma unroll
        for (int u = 0; u < 8; ++u) gt[u] = Raw<T>::get(gv, u);
      }
    }
    if (p.bias != nullptr) {
      if (pre) {  // float32, already multiplied by the gate, one vector per gate vector
        const float* bp = bias_f + grow + n;
        const f32x4_v b0 = *reinterpret_cast<const f32x4_v*>(bp), b1 = *reinterpret_cast<const f32x4_v*>(bp + 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) { bs[u] = b0[u]; bs[4 + u] = b1[u]; }
      } else {
        const u32x4 bv = load_raw(bias_h + n);
#pragma unroll
        for (int u = 0; u < 8; ++u) bs[u] = gt[u] * Raw<T>::get(bv, u);
      }
    }
    const u32x4 rv = load_raw(static_cast<const T*>(p.residual) + m * p.ldr + n);
#pragma unroll
    for (int u = 0; u < 8; ++u) y[u] = gemm_clipped<T>(p, fmaf(gt[u], y[u], bs[u]) + Raw<T>::get(rv, u));
  } else {
    if (p.bias != nullptr) {
      const u32x4 bv = load_raw(bias_h + n);
#pragma unroll
      for (int u = 0; u < 8; ++u) y[u] += Raw<T>::get(bv, u);
    }
    if (gelu) {
#pragma unroll
      for (int u = 0; u < 8; ++u) y[u] = gemm_gelu_tanh(y[u]);
    }
  }
  u32x4 o;
#pragma unroll
  for (int u = 0; u < 4; ++u) Raw<T>::set2(o, u, y[2 * u], y[2 * u + 1]);
  store_raw(static_cast<T*>(p.out) + m * p.ldo + n, o);
}

inline GemmEpilogue gemm_epilogue_of(const GemmCall& c) {
  GemmEpilogue e;
  e.bias = c.bias; e.residual = c.residual; e.gate = c.gate; e.out = c.out;
  e.M = c.M; e.N = c.N; e.ldo = c.ldo; e.ldr = c.ldr; e.ldg = c.ldg;
  e.epilogue = c.epilogue; e.gate_f32 = c.gate_f32; e.rows_per_gate = c.rows_per_gate;
  e.most = c.clip ? 65504.f : INFINITY;
  return e;
}

}  // namespace odit
