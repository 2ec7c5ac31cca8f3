// LayerNorm without affine, modulation and projection to few features in one launch: a model's head,
//     y = (norm(x) (1 + scale) + shift) W^T + b,
// whose W is read by everyone (64 features of 3072: 393 KB) and whose rows are read once.
//
// Workgroup: 8 wavefronts on a tile of 16 rows x 16 F features, each with an eighth of the reduction, which goes from global memory straight into
// the registers that v_mfma_f32_16x16x32 reads it from: all of a wavefront's rows and its first steps of W are asked for at once, and nothing is
// waited for but the rows. A lane has one row of a fragment, so the sums of the norm go over its own elements, the four lanes of the row and,
// through LDS, the wavefronts; the norm's operations are adaln_rows_kernel's, in another order of the sums. The normed values, rounded as that
// kernel stores them, are the matrix operand in their place. The wavefronts' sums meet in LDS, added in their order.
//
// What bounds it: what a CU fetches (52 KB/us: 196 KB for a tile of 16 x 16 at K=3072, 3.8 us) and the norm's arithmetic, 12 operations an element
// on 96 elements a lane (4 us), around a chain of two barriers. Two row fragments or 16 wavefronts to a workgroup are slower at every size (32 x 32
// features 23 us, 16 wavefronts 12.3, where this takes 10.3: 512 rows, K=3072). In the place of two launches, the norm's and the tile kernel's, of
// which that one has a workgroup for every 128 rows and 48 steps to go (17.2 us at 256 rows, 22 at 4096).
#include "gemm_epilogue.h"

namespace odit {

namespace {

constexpr int kHeadWaves = 8;

struct HeadParams {
  const void *x, *w, *bias, *shift, *scale;
  void* out;
  int M, N, S, n_tiles;
  uint32_t ldx, ldw, x_bytes, w_bytes;  // bytes
  int64_t ldo, mod_stride;
  float eps;
};

// NS: steps of 32 of a wavefront's part of the reduction (K = 256 NS); PRE: steps of W that are on their way
template <typename T, int NS, int F, int PRE>
__global__ __launch_bounds__(64 * kHeadWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void linear_head_kernel(const HeadParams p) {
  using M = Mma16<T>;
  using frag = typename M::frag;
  constexpr int kAhead = 4;  // steps of shift and scale
  __shared__ __attribute__((aligned(16))) float part[16][kHeadWaves][2];
  __shared__ __attribute__((aligned(16))) f32x4_v red[kHeadWaves][F][64];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int mt = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(t) / static_cast<unsigned>(p.n_tiles));
  const int m = mt * 16 + l16, n0 = (t - mt * p.n_tiles) * (16 * F);
  const int k = wave * (NS * 32) + lq * 8;
  const auto xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, static_cast<int>(p.x_bytes), 0x00020000);
  const auto ws = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.w), 0, static_cast<int>(p.w_bytes), 0x00020000);

  // (rows and features past the end: zeros, from past the operand's end)
  const uint32_t xat = static_cast<uint32_t>(m) * p.ldx;
  const float k0 = to_float(__builtin_bit_cast(T, static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(xs, xat, 0, 0))));
  u32x4 x[NS], w[PRE][F];
#pragma unroll
  for (int i = 0; i < NS; ++i) x[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, xat + k * 2 + i * 64, 0, 0));
  uint32_t wat[F];
#pragma unroll
  for (int f = 0; f < F; ++f) {
    // (of two accumulators the features alternate by fours: a lane ends up with 8 consecutive ones)
    const int row = F == 1 ? l16 : 32 * (f / 2) + ((l16 >> 2) << 3) + (f % 2) * 4 + (l16 & 3);
    wat[f] = static_cast<uint32_t>(n0 + row) * p.ldw + k * 2;
  }
  auto ask_w = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < F; ++f) w[i % PRE][f] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ws, wat[f] + i * 64, 0, 0));
  };
#pragma unroll
  for (int i = 0; i < PRE; ++i) ask_w(i);
  __builtin_amdgcn_sched_barrier(0);

  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float d = Raw<T>::get(x[i], u) - k0;
      s1 += d;
      s2 = fmaf(d, d, s2);
    }
  s1 += __shfl_xor(s1, 16);
  s2 += __shfl_xor(s2, 16);
  s1 += __shfl_xor(s1, 32);
  s2 += __shfl_xor(s2, 32);
  if (lq == 0) {
    part[l16][wave][0] = s1;
    part[l16][wave][1] = s2;
  }
  __syncthreads();
  s1 = s2 = 0.f;
#pragma unroll
  for (int i = 0; i < kHeadWaves / 2; ++i) {
    const f32x4_v v = *reinterpret_cast<const f32x4_v*>(&part[l16][2 * i][0]);
    s1 += v[0] + v[2];
    s2 += v[1] + v[3];
  }
  constexpr float kInv = 1.f / static_cast<float>(256 * NS);
  const float m1 = s1 * kInv, mean = k0 + m1, rstd = rsqrtf(fmaxf(s2 * kInv - m1 * m1, 0.f) + p.eps);
  const int64_t mod = static_cast<int64_t>(static_cast<unsigned>(m < p.M ? m : p.M - 1) / static_cast<unsigned>(p.S)) * p.mod_stride + k;
  u32x4 scale[kAhead], shift[kAhead];
  auto ask = [&](int i) __attribute__((always_inline)) {
    scale[i % kAhead] = load_raw(static_cast<const T*>(p.scale) + mod + i * 32);
    shift[i % kAhead] = load_raw(static_cast<const T*>(p.shift) + mod + i * 32);
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) ask(i);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const u32x4 raw = x[i], sc = scale[i % kAhead], sh = shift[i % kAhead];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      Raw<T>::set2(x[i], u, fmaf((Raw<T>::get(raw, 2 * u) - mean) * rstd, 1.f + Raw<T>::get(sc, 2 * u), Raw<T>::get(sh, 2 * u)),
                   fmaf((Raw<T>::get(raw, 2 * u + 1) - mean) * rstd, 1.f + Raw<T>::get(sc, 2 * u + 1), Raw<T>::get(sh, 2 * u + 1)));
    if (i + kAhead < NS) ask(i + kAhead);
  }

  f32x4_v acc[F];
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] = f32x4_v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NS; ++i) {
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = M::run(__builtin_bit_cast(frag, w[i % PRE][f]), __builtin_bit_cast(frag, x[i]), acc[f]);
    if (i + PRE < NS) ask_w(i + PRE);
  }
#pragma unroll
  for (int f = 0; f < F; ++f) red[wave][f][lane] = acc[f];
  __syncthreads();

  constexpr int kPer = F == 1 ? 1 : 2;  // accumulators to a lane's consecutive features
  if (wave >= F / kPer) return;
  f32x4_v y[kPer];
#pragma unroll
  for (int a = 0; a < kPer; ++a) {
    y[a] = red[0][wave * kPer + a][lane];
#pragma unroll
    for (int o = 1; o < kHeadWaves; ++o) y[a] += red[o][wave * kPer + a][lane];
  }
  const int n = n0 + wave * (16 * kPer) + lq * (4 * kPer);
  if (m >= p.M || n >= p.N) return;
  T* const out = static_cast<T*>(p.out) + m * p.ldo + n;
  const T* const bias = p.bias != nullptr ? static_cast<const T*>(p.bias) + n : nullptr;
  if constexpr (kPer == 2) {
    const u32x4 b = bias != nullptr ? load_raw(bias) : u32x4{0u, 0u, 0u, 0u};
    u32x4 o;
#pragma unroll
    for (int u = 0; u < 4; ++u) Raw<T>::set2(o, u, y[u >> 1][2 * (u & 1)] + Raw<T>::get(b, 2 * u), y[u >> 1][2 * (u & 1) + 1] + Raw<T>::get(b, 2 * u + 1));
    store_raw(out, o);
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) out[u] = from_float<T>(y[0][u] + (bias != nullptr ? to_float(bias[u]) : 0.f));
  }
}

template <typename T, int NS>
void go(HeadParams& p, int features, hipStream_t stream) {
  p.n_tiles = (p.N + features - 1) / features;
  const dim3 grid(static_cast<unsigned>((p.M + 15) / 16 * p.n_tiles)), block(64 * kHeadWaves);
  if (features == 16) hipLaunchKernelGGL((linear_head_kernel<T, NS, 1, NS>), grid, block, 0, stream, p);
  else if (features == 32) hipLaunchKernelGGL((linear_head_kernel<T, NS, 2, NS>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((linear_head_kernel<T, NS, 4, 4>), grid, block, 0, stream, p);
}

// Features to a tile: a round of workgroups (one to a CU) costs what it fetches, 16 rows and the tile's features, and the norm, which every tile of the same
// rows does again. us at K=3072, N=64, 16 / 32 / 64 features: 256 rows 10.1 / 12.3 / 17.2, 1024 10.6 / 12.6 / 17.5, 1500 19.5 / 12.7 / 17.6, 4096
// 38 / 24 / 17.9, 8192 72 / 46 / 34; K=1024: 512 rows 5.4 / 5.5 / 7.3, 4096 19 / 10.5 / 7.9. 0: none in up to two rounds, and the norm and the
// projection in launches of their own are as fast (16000 rows 66 in four rounds, 61 in two launches; 8192 34 and 43, 4096 18 and 33, 1024 10.6 and 22.6,
// 256 10.1 and 20.3).
int head_features(int M, int N, int K, int cus) {
  const float k = static_cast<float>(K) / 1024.f, round[3] = {2.3f + 2.3f * k, 1.9f + 3.1f * k, 1.9f + 4.7f * k};
  int best = 0;
  float us = 0.f;
  for (int i = 0; i < 3; ++i) {
    const int64_t tiles = static_cast<int64_t>((M + 15) / 16) * ((N + (16 << i) - 1) / (16 << i)), rounds = (tiles + cus - 1) / cus;
    if (rounds > 2 || (best != 0 && rounds * round[i] >= us)) continue;
    best = 16 << i;
    us = rounds * round[i];
  }
  return best;
}

}  // namespace

// K: the kernel is made for multiples of 256, a step's fragments of 8 wavefronts, and built for the three that the times above were taken at; heads of other widths keep their
// two launches. What a tuning call found for the projection alone is not asked: the norm in front of it is a launch of its own there (6 us and more of the 10 to 34).
int linear_head_features(const GemmCall& c, const RowNorm& n, int dtype, int cus) {
  if ((c.K != 1024 && c.K != 2048 && c.K != 3072) || c.N > 64 || cus <= 0 || !gemm_streamk_takes(c, dtype) || !aligned16(n.shift) || !aligned16(n.scale) ||
      n.stride % 8 != 0 || (c.epilogue != ODIT_EPI_NONE && c.epilogue != ODIT_EPI_BIAS) || !gemm_rows_fit(c.M + 16, c.ldx, c.K) || !gemm_rows_fit(c.N + 64, c.ldw, c.K))
    return 0;
  return head_features(c.M, c.N, c.K, cus);
}

int launch_linear_head(const GemmCall& c, const RowNorm& n, int features, int dtype, hipStream_t stream) {
  HeadParams p;
  p.x = c.x; p.w = c.w; p.bias = c.epilogue == ODIT_EPI_BIAS ? c.bias : nullptr; p.shift = n.shift; p.scale = n.scale; p.out = c.out;
  p.M = c.M; p.N = c.N; p.S = n.S;
  p.ldx = static_cast<uint32_t>(c.ldx * 2); p.ldw = static_cast<uint32_t>(c.ldw * 2);
  p.x_bytes = static_cast<uint32_t>((static_cast<uint64_t>(c.M - 1) * c.ldx + c.K) * 2);
  p.w_bytes = static_cast<uint32_t>((static_cast<uint64_t>(c.N - 1) * c.ldw + c.K) * 2);
  p.ldo = c.ldo; p.mod_stride = n.stride; p.eps = n.eps;
#define ODIT_HEAD(NS) do { if (dtype == ODIT_BF16) go<bf16_t, NS>(p, features, stream); else go<f16_t, NS>(p, features, stream); } while (0)
  if (c.K == 1024) ODIT_HEAD(4);
  else if (c.K == 2048) ODIT_HEAD(8);
  else ODIT_HEAD(12);
#undef ODIT_HEAD
  return check_launch("odit_linear_norm (head)");
}

}  // namespace odit
