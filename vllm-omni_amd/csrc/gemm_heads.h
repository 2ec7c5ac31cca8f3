// Query, key and value heads at the end of a GEMM tile (gemm_tile.h, gemm_small.h): what is done to the 8 consecutive features that a
// lane holds of a row, and where they go.
#pragma once

#include "gemm_epilogue.h"

namespace odit {

// s of this lane and of the one 16 (32) further or before: the swap of two copies of s leaves one's lanes in each half's pairs
template <typename Pair> __device__ __forceinline__ float add_swapped(float, Pair p) { return __uint_as_float(p[0]) + __uint_as_float(p[1]); }

// Where this lane's rows r, r + 16, ... of a tile go, and their rotary factors of in-head features d .. d + 7
template <int MH>
struct HeadRows {
  int at[MH];  // row of the outputs, -1: none
  f32x4_v cos[MH], sin[MH];
  __device__ __forceinline__ void ask(const HeadsOut& h, int M, int m0, int r, int d) {
#pragma unroll
    for (int i = 0; i < MH; ++i) {
      const int row = m0 + r + i * 16, m = row < M ? row : M - 1;
      const int b = h.div_mul == 0 ? m : static_cast<int>(__umulhi(m, h.div_mul) >> h.div_shift), s = m - b * h.S;
      at[i] = row < M ? b * h.S_total + h.offset + s : -1;
      const int64_t t = static_cast<int64_t>(s) * (h.D / 2) + d / 2;
      cos[i] = *reinterpret_cast<const f32x4_v*>(h.cos + t);
      sin[i] = *reinterpret_cast<const f32x4_v*>(h.sin + t);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// 8 features of a query or key: norm (rstd of the head's row), weight and rotation in pairs, the operations of qknorm_flat_kernel: its
// bits, but for which of an odd feature's two products the compiler rounds (f16: 6 elements in 100000 differ, by a step).
template <typename T> __device__ __forceinline__ u32x4 turn_head(u32x4 v, float rstd, u32x4 weight, f32x4_v cos, f32x4_v sin) {
  u32x4 o;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float x0 = Raw<T>::get(v, 2 * u) * rstd * Raw<T>::get(weight, 2 * u), x1 = Raw<T>::get(v, 2 * u + 1) * rstd * Raw<T>::get(weight, 2 * u + 1);
    Raw<T>::set2(o, u, x0 * cos[u] - x1 * sin[u], x1 * cos[u] + x0 * sin[u]);
  }
  return o;
}

// m / S as a multiply-high and a shift, exact for m < 2^31: l = ceil(log2 S), mul = ceil(2^(31 + l) / S). (One row to a batch entry:
// mul 0, the row number is the entry's.)
inline void fill_heads_division(HeadsOut& h) {
  h.div_mul = h.div_shift = 0;
  if (h.q == nullptr || h.S <= 1) return;
  uint32_t l = 1;
  while ((1ull << l) < static_cast<uint64_t>(h.S)) ++l;
  h.div_mul = static_cast<uint32_t>(((1ull << (31 + l)) + h.S - 1) / h.S);
  h.div_shift = l - 1;
}

}  // namespace odit
