// 16-bit GEMM y = x W^T for products that are small altogether (models of a few hundred channels), one problem or two of the same
// N and K in one launch: one 64 x 64 output tile per workgroup of 8 wavefronts, no reduction is divided.
//
// What bounds it: latency. A launch of some dozens of workgroups is one chain of arguments, first loads, matrix work, epilogue
// operands and stores; at these sizes the work itself takes a microsecond. So everything that does not depend on the product is
// asked for at once: bias, gate and residual go to registers and up to 8 steps of both operands (64 x 64 pieces of x and of W,
// global memory straight into LDS, 16 KB a step) are in flight before anything is waited for, and the tile is stored from
// registers. The stream-K kernel, which cuts reductions of four steps over several workgroups, spends most of its time on the
// hand-over there. us, stream-K / this kernel: M=256+64, K=256: N=768 13.7 / 5.3, N=256 13.0 / 4.5, N=1024 with GELU 14.9 / 5.9;
// N=256, K=1024 21.5 / 7.8. One problem, the library / this kernel: M=64, N=256, K=256 9.0 / 5.2.
//
// Two wavefronts to a SIMD, which issue while the other one waits: a wavefront alone issues a vector instruction every 7 to 8 cycles, and
// addresses, first fragments and the epilogue's arithmetic are in the chain. us a launch in a row, 4 wavefronts (32 x 32 outputs each) / 8, the
// same bits: M=64 N=64 K=256 4.06 / 3.41; M=128 N=768 K=256 4.31 / 3.64; M=320 N=1024 K=256 with GELU 4.95 / 3.92; M=1024 N=1024 K=1024 with
// GELU 8.35 / 7.26; 1024 tiles of K=64 5.81 / 5.69, of K=128 with GELU 7.44 / 6.66; 512 of K=256 5.50 / 5.02.
//
// A wavefront owns 16 rows x 32 features as two accumulators of v_mfma_f32_16x16x32 with W rows as the A operand; the features
// of the two accumulators interleave by 4, so that a lane ends up with 8 consecutive ones of a row. Chunks of 16 bytes are
// XORed with bits of the row as in gemm_tile.h. One barrier per step.
//
// NORM: the rows are normed (and modulated) on the way (adaln_rows_kernel's operations, its bits), for reductions whose steps are all in LDS
// at once. A launch of that kernel in front is 2.3 to 2.5 us one after the other, for a microsecond of work that every workgroup can do for
// the 64 rows it reads anyway (1.7 us more of a launch): each wavefront norms the 8 rows that it has fetched itself, eight lanes to a
// row, so nothing is waited for that was not before.
#pragma once

#include "gemm_epilogue.h"
#include "gemm_heads.h"

namespace odit {

namespace {

constexpr int kSmallWaves = 8, kSmallTile = 64, kSmallStages = 8, kSmallPiece = kSmallTile * kGemmBK * 2, kSmallStage = 2 * kSmallPiece;

// kNormAll: LayerNorm and modulation of the rows of every problem. kNormStem: of two problems with reductions of their own the second one's rows
// are RMS-normed and weighted (head_norm_kernel's operations, its bits), the first one's as they are.
constexpr int kNormAll = 1, kNormStem = 2;

struct SmallProblem {
  const void *x, *w;
  int M;
  uint32_t ldx, ldw;  // bytes
  uint32_t x_bytes, w_bytes;
  GemmEpilogue ep;
};

struct SmallParams {
  SmallProblem q[2];
  int N, k_steps, n_tiles;
  int tiles0;  // of the first problem
};

template <bool HEADS> struct SmallHeads : SmallParams {};
template <> struct SmallHeads<true> : SmallParams {
  HeadsOut heads[2];  // of 64 features: a tile is one head
};
template <bool HEADS, int NORM> struct SmallArgs : SmallHeads<HEADS> {};
template <bool HEADS> struct SmallArgs<HEADS, kNormAll> : SmallHeads<HEADS> {
  RowNorm norm[2];
};
template <> struct SmallArgs<false, kNormStem> : SmallParams {
  const void* weight;  // of the second problem's norm
  float eps;
  int k_steps1;  // the second problem's
};

typedef __attribute__((address_space(3))) void* lds_void_p;

// The wavefront's 8 rows of the tile, whose pieces it has asked for: LayerNorm and modulation in place. `ask` asks for what comes behind
// them. Lane l works on row l / 8, chunk l % 8 of every step: the sums over a row go chunk by chunk, over the 8 lanes, by twos of steps, and up
// from there: the order of adaln_rows_kernel's wavefront with a chunk to a lane.
template <typename T, int S, typename Ask>
__device__ __forceinline__ void norm_rows(const RowNorm& nm, char* lds, int m0, int M, int nk, int wave, int lane, Ask&& ask) {
  const int r = wave * 8 + (lane >> 3), j = lane & 7, C = nk * kGemmBK;
  const int m = m0 + r < M ? m0 + r : M - 1;
  const int64_t at = static_cast<int64_t>(static_cast<unsigned>(m) / static_cast<unsigned>(nm.S)) * nm.stride + j * 8;
  u32x4 scale[S], shift[S], raw[S];
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < nk) {
      scale[i] = load_raw(static_cast<const T*>(nm.scale) + at + i * kGemmBK);
      shift[i] = load_raw(static_cast<const T*>(nm.shift) + at + i * kGemmBK);
    }
  ask();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int turn = (r >> 1) & 7;
  auto chunk = [&](int i) { return lds + i * kSmallStage + r * 128 + ((j ^ turn) << 4); };
  const float k0 = to_float(*reinterpret_cast<const T*>(lds + r * 128 + (turn << 4)));
  float s1[S], s2[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    s1[i] = s2[i] = 0.f;
    if (i < nk) {
      raw[i] = *reinterpret_cast<const u32x4*>(chunk(i));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float d = Raw<T>::get(raw[i], u) - k0;
        s1[i] += d;
        s2[i] = fmaf(d, d, s2[i]);
      }
      s1[i] = row_group_sum<8>(s1[i]);
      s2[i] = row_group_sum<8>(s2[i]);
    }
  }
  float a1 = 0.f, a2 = 0.f;
#pragma unroll
  for (int i = 0; i < S; i += 2) {
    a1 += s1[i] + (i + 1 < S ? s1[i + 1 < S ? i + 1 : i] : 0.f);
    a2 += s2[i] + (i + 1 < S ? s2[i + 1 < S ? i + 1 : i] : 0.f);
  }
  const float inv_c = 1.f / static_cast<float>(C);
  const float m1 = a1 * inv_c;
  const float mean = k0 + m1;
  const float rstd = rsqrtf(fmaxf(a2 * inv_c - m1 * m1, 0.f) + nm.eps);
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < nk) {
      u32x4 o;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        Raw<T>::set2(o, u, fmaf((Raw<T>::get(raw[i], 2 * u) - mean) * rstd, 1.f + Raw<T>::get(scale[i], 2 * u), Raw<T>::get(shift[i], 2 * u)),
                     fmaf((Raw<T>::get(raw[i], 2 * u + 1) - mean) * rstd, 1.f + Raw<T>::get(scale[i], 2 * u + 1), Raw<T>::get(shift[i], 2 * u + 1)));
      *reinterpret_cast<u32x4*>(chunk(i)) = o;
    }
}

// RMSNorm and weight of the same rows, a power of two of steps: the sums go over the lanes of a row in head_norm_kernel's order
template <typename T, int S, typename Ask>
__device__ __forceinline__ void rms_rows(const void* weight, float eps, char* lds, int nk, int wave, int lane, Ask&& ask) {
  const int r = wave * 8 + (lane >> 3), j = lane & 7, turn = (r >> 1) & 7;
  u32x4 w[S], raw[S];
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < nk) w[i] = load_raw(static_cast<const T*>(weight) + j * 8 + i * kGemmBK);
  ask();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  auto chunk = [&](int i) { return lds + i * kSmallStage + r * 128 + ((j ^ turn) << 4); };
  float sq[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    sq[i] = 0.f;
    if (i < nk) {
      raw[i] = *reinterpret_cast<const u32x4*>(chunk(i));
#pragma unroll
      for (int u = 0; u < 8; ++u) sq[i] = fmaf(Raw<T>::get(raw[i], u), Raw<T>::get(raw[i], u), sq[i]);
      sq[i] = row_group_sum<8>(sq[i]);
    }
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < S; i += 2) sum += sq[i] + (i + 1 < S ? sq[i + 1 < S ? i + 1 : i] : 0.f);
  const float rstd = rsqrtf(sum * (1.f / static_cast<float>(nk * kGemmBK)) + eps);
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < nk) {
      u32x4 o;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        Raw<T>::set2(o, u, Raw<T>::get(raw[i], 2 * u) * rstd * Raw<T>::get(w[i], 2 * u), Raw<T>::get(raw[i], 2 * u + 1) * rstd * Raw<T>::get(w[i], 2 * u + 1));
      *reinterpret_cast<u32x4*>(chunk(i)) = o;
    }
}

// S: stages (as many as there are steps where those are fewer than 8: several workgroups to a CU)
// HEADS: query, key and value heads of 64 features (gemm_heads.h), a tile each
template <typename T, int S, bool HEADS, int NORM>
__global__ __launch_bounds__(64 * kSmallWaves) void gemm_small_kernel(const SmallArgs<HEADS, NORM> p) {
  using M = Mma16<T>;
  using frag = typename M::frag;
  __shared__ __attribute__((aligned(1024))) char lds[S * kSmallStage];
  __shared__ float squares[HEADS ? kSmallTile * 2 : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;
  const int l16 = lane & 15, lq = lane >> 4;
  const int which = static_cast<int>(blockIdx.x) >= p.tiles0 ? 1 : 0;
  const SmallProblem& q = p.q[which];
  const int t = static_cast<int>(blockIdx.x) - (which ? p.tiles0 : 0);
  const int mt = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(t) / static_cast<unsigned>(p.n_tiles));
  const int m0 = mt * kSmallTile, n0 = (t - mt * p.n_tiles) * kSmallTile;
  int nk = p.k_steps;
  if constexpr (NORM == kNormStem) nk = which ? p.k_steps1 : nk;

  auto make_rsrc = [](const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    u32x4_v r;
    r.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    r.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32) & 0xffffu);
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;
    return r;
  };
  const u32x4_v xr = make_rsrc(q.x, q.x_bytes), wr = make_rsrc(q.w, q.w_bytes);

  // this wavefront's share of a piece is rows 8 wave .. + 7, one instruction; rows past the end re-read the last one
  const int r = wave * 8 + (lane >> 3), ch = lane & 7;
  const int rx = m0 + r < q.M ? m0 + r : q.M - 1, rw = n0 + r < p.N ? n0 + r : p.N - 1;
  const uint32_t vx = static_cast<uint32_t>(rx) * q.ldx + static_cast<uint32_t>((ch ^ ((r >> 1) & 7)) << 4);
  const uint32_t vw = static_cast<uint32_t>(rw) * q.ldw + static_cast<uint32_t>((ch ^ (((r >> 1) & 1) | (((r >> 3) & 3) << 1))) << 4);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_p)lds)) + wave * 1024;
  auto load = [&](uint32_t dst, uint32_t off, u32x4_v rs, int soff) {
    load_lds16(__builtin_amdgcn_readfirstlane(dst), off, rs, __builtin_amdgcn_readfirstlane(soff));
  };
  auto issue_x = [&](int i, int stage) { load(lds0 + stage * kSmallStage, vx, xr, i * (kGemmBK * 2)); };
  auto issue_w = [&](int i, int stage) { load(lds0 + stage * kSmallStage + kSmallPiece, vw, wr, i * (kGemmBK * 2)); };
  auto issue = [&](int i, int stage) {
    issue_x(i, stage);
    issue_w(i, stage);
  };

  // operands of the epilogue: row m, features n .. n + 7
  const GemmEpilogue& e = q.ep;
  const int m = m0 + wm * 16 + l16, n = n0 + wn * 32 + lq * 8;
  const bool gated = e.epilogue == ODIT_EPI_GATED_RESIDUAL || e.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
  const bool gelu = e.epilogue == ODIT_EPI_GELU_TANH || e.epilogue == ODIT_EPI_BIAS_GELU_TANH;
  float gt[8], bs[8];
  u32x4 res = {};
  HeadRows<1> rows;
  u32x4 bias = {0u, 0u, 0u, 0u}, weight = bias;
  int third = 0;
  if constexpr (HEADS) {
    const HeadsOut& h = p.heads[which];
    third = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(n0) / static_cast<unsigned>(h.HD));
    if (e.bias != nullptr) bias = load_raw(static_cast<const T*>(e.bias) + n);
    if (third < 2) weight = load_raw(static_cast<const T*>(third == 0 ? h.wq : h.wk) + (n - n0));
    rows.ask(h, q.M, m0, wm * 16 + l16, n - n0);
  } else {
    const int row = m < q.M ? m : q.M - 1, col = n < p.N ? n : 0;
    gemm_epilogue_vectors8<T>(e, row, col, gt, bs);
    if (gated) res = load_raw(static_cast<const T*>(e.residual) + row * e.ldr + col);
  }
  auto issue_first = [&](auto&& one) {
#pragma unroll
    for (int d = 0; d < S; ++d)
      if (d < nk) one(d, d);
  };
  if constexpr (NORM == kNormAll) {
    issue_first(issue_x);
    norm_rows<T, S>(p.norm[which], lds, m0, q.M, nk, wave, lane, [&] { issue_first(issue_w); });
  } else if constexpr (NORM == kNormStem) {
    issue_first(issue_x);
    if (which) rms_rows<T, S>(p.weight, p.eps, lds, nk, wave, lane, [&] { issue_first(issue_w); });
    else issue_first(issue_w);
  } else {
    issue_first(issue);
  }

  const int xrow = wm * 16 + l16;
  const int xa = xrow * 128 + ((lq ^ ((xrow >> 1) & 7)) << 4);
  const int wrow = wn * 32 + ((l16 >> 2) << 3) + (l16 & 3);
  const int wa = kSmallPiece + wrow * 128 + ((lq ^ (((wrow >> 1) & 1) | (((wrow >> 3) & 3) << 1))) << 4);
  f32x4_v acc[2] = {f32x4_v{0.f, 0.f, 0.f, 0.f}, f32x4_v{0.f, 0.f, 0.f, 0.f}};
  for (int i = 0; i < nk; ++i) {
    // this wavefront's loads of step i have landed and its reads of step i - 1 are in registers; behind the barrier that holds for
    // every wavefront, and the stage of step i - 1 is free
    if (S == kSmallStages && i + S - 2 < nk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kSmallStages - 2) * 2) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (S == kSmallStages && i > 0 && i - 1 + S < nk) issue(i - 1 + S, (i - 1) % S);
    const char* st = lds + (i % S) * kSmallStage;
    frag xf[2], wf[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      xf[ks] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(st + (xa ^ (ks * 64))));
#pragma unroll
      for (int b = 0; b < 2; ++b) wf[ks][b] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(st + (wa ^ (ks * 64)) + b * 512));
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[b] = M::run(wf[ks][b], xf[ks], acc[b]);
  }

  if constexpr (HEADS) {
    const HeadsOut& h = p.heads[which];
    const int r = wm * 16 + l16;
    u32x4 x;
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      Raw<T>::set2(x, u, acc[u / 2][2 * (u % 2)] + Raw<T>::get(bias, 2 * u), acc[u / 2][2 * (u % 2) + 1] + Raw<T>::get(bias, 2 * u + 1));
#pragma unroll
    for (int u = 0; u < 8; ++u) s = fmaf(Raw<T>::get(x, u), Raw<T>::get(x, u), s);
    s = add_swapped(s, __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false));
    s = add_swapped(s, __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false));
    squares[r * 2 + wn] = s;  // (the same from four lanes)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    void *qo = h.q, *ko = h.k, *vo = h.v;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+s"(qo), "+s"(ko), "+s"(vo));  // (values of their own: the choice by `third` would be an index into a copy of them in memory)
#endif
    T* const out = static_cast<T*>(third == 0 ? qo : third == 1 ? ko : vo) + (n - third * h.HD);
    if (third < 2) {
      const float rstd = rsqrtf((squares[r * 2] + squares[r * 2 + 1]) * (1.f / 64) + h.eps);
      x = turn_head<T>(x, rstd, weight, rows.cos[0], rows.sin[0]);
    }
    if (rows.at[0] >= 0) store_raw(out + static_cast<int64_t>(rows.at[0]) * h.HD, x);
    return;
  }
  if (m >= q.M || n >= p.N) return;
  u32x4 o;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float y[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int f = 2 * u + t;
      const float a = acc[f / 4][f % 4];
      y[t] = gated ? gemm_clipped<T>(e, fmaf(gt[f], a, bs[f]) + Raw<T>::get(res, f)) : a + bs[f];
      if (!gated && gelu) y[t] = gemm_gelu_tanh(y[t]);
    }
    Raw<T>::set2(o, u, y[0], y[1]);
  }
  store_raw(static_cast<T*>(e.out) + m * e.ldo + n, o);
}

inline void fill_small_params(SmallParams& p, const GemmCall* c, int count, int (&tiles)[2]) {
  p.N = c[0].N;
  p.n_tiles = (p.N + kSmallTile - 1) / kSmallTile;
  p.k_steps = c[0].K / kGemmBK;
  for (int i = 0; i < 2; ++i) {
    const GemmCall& g = c[i < count ? i : 0];
    SmallProblem& q = p.q[i];
    q.x = g.x; q.w = g.w; q.M = g.M;
    q.ldx = static_cast<uint32_t>(g.ldx * 2); q.ldw = static_cast<uint32_t>(g.ldw * 2);
    q.x_bytes = static_cast<uint32_t>((static_cast<uint64_t>(g.M - 1) * g.ldx + g.K) * 2);
    q.w_bytes = static_cast<uint32_t>((static_cast<uint64_t>(g.N - 1) * g.ldw + g.K) * 2);
    q.ep = gemm_epilogue_of(g);
    if (i < count) tiles[i] = (g.M + kSmallTile - 1) / kSmallTile * p.n_tiles;
  }
  p.tiles0 = tiles[0];
}

}  // namespace

}  // namespace odit
