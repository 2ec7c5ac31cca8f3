// Projections of a few rows (M <= 16): the timestep embedding, the modulation parameters of all blocks from one stacked
// weight, the head's norm. out[M,N] = act(x)[M,K] W[N,K]^T + bias, act = identity or SiLU rounded to the tensor type.
//
// Bound: the weights are read once (N K 2 bytes: 453 MB for two blocks of width 3072) and everything else is noise, so
// the kernels are weight streams with enough loads in flight. Loads are non-temporal: without, the weights push activations out of
// the last-level cache and wait for their write-back. What a stream reaches hangs on what one load covers, measured by loads alone
// (TB/s, N=442368, K=3072, non-temporal / not): 1 KB of one row 7.0 / 6.2, 64 bytes of each of 16 rows 5.6 / 6.4.
//
// linear_stream_kernel, up to 4 rows, K a multiple of 512: a load of a wavefront is 1 KB of one row of W, two or four rows at a
// time, double-buffered (24 wavefronts a CU with 4 to 8 KB each in flight). A lane multiplies its 8 weights with the same 8
// elements of every row of x (from LDS, activated once) in float32, 8 M fused multiply-adds a load; a row's 64 partial sums
// meet by DPP behind its last chunk. With 4 rows of x the vector unit is half busy; past that the matrix kernel is the better
// one. us and TB/s from cold caches, linear_few_kernel / this: N=442368, K=3072, one row 515 (5.3) / 397 (6.9), two 521 / 405, four
// 534 / 440; N=73728 two rows 90 / 68; N=18432 27 / 20.5; N=6144 13.2 / 10.0; N=3072 8.8 / 7.1; N=30720, K=5120 72 / 50.
//
// linear_few_kernel, the others. A workgroup of 8 waves takes 16 features at a time; the waves divide the reduction. A wave loads 16
// features x 32 reduction elements with one 16-byte load per lane, straight into the A operand of v_mfma_f32_16x16x32 (lane l:
// feature l % 16, elements 8 (l / 16) ..); adjacent loads of a wave cover the rest of the lines. kSteps loads are in flight while the
// kSteps before them are multiplied, across the end of a tile too: the grid is persistent (3 workgroups per CU, tiles strided
// over the grid) and the only thing a tile's end costs is one barrier. x sits in LDS (rows 16 bytes apart beyond their
// length: conflict-free), is the B operand (column = row of x; columns past M repeat the last row and are not stored), and is
// activated once while it is staged. The 8 partial sums of a tile meet in LDS (two buffers by turns, so one barrier per
// tile), in the order of the waves: results do not depend on timing.
//
// Both take two weights in one launch, the second one's features behind the first one's: the modulation parameters of all blocks and the
// head's norm follow from the same rows. us, two launches / one, cold weights, two rows: K=3072, 442368 + 6144 features 429.7 / 427.2,
// 73728 + 6144 81.3 / 78.2, 18432 + 6144 30.7 / 26.5; K=256, 24576 + 512 14.3 / 11.2, 6144 + 512 9.4 / 5.6.
// linear_few_sinusoid_kernel: the rows of x are a timestep's cosines and sines, formed where they are staged (time_sinusoid_kernel's
// operations): 3072 features, K=256 5.8 / 4.3, the launch less.
#include <type_traits>

#include "odit_common.h"
#include "gemm_bf16.h"
#include "time_sinusoid.h"
#include "time_tokens.h"

namespace odit {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T> __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mfma16<bf16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x4 mfma16<f16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

constexpr int kWaves = 8, kTile = 16, kStepK = 32, kSteps = 4;
constexpr int kRedBytes = 2 * kWaves * 64 * 16;

template <typename T> __device__ __forceinline__ u32x4 silu8(u32x4 r) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = Raw<T>::get(r, 2 * p), b = Raw<T>::get(r, 2 * p + 1);
    Raw<T>::set2(r, p, a / (1.f + __expf(-a)), b / (1.f + __expf(-b)));
  }
  return r;
}

// x, activated, to LDS: `rows` rows of `vecs` 16-byte vectors, `pitch` apart
template <typename T, bool SILU>
__device__ __forceinline__ void stage_rows(const T* __restrict__ x, u32x4* xs, int rows, int vecs, int pitch, int64_t ldx) {
  for (int i = threadIdx.x; i < rows * vecs; i += kWaves * 64) {
    const int m = i / vecs, v = i - m * vecs;
    const u32x4 r = load_raw(x + m * ldx + v * 8);
    xs[m * pitch + v] = SILU ? silu8<T>(r) : r;
  }
}

// A weight and where its products go
template <typename T> struct FewOut {
  const T *w, *bias;
  T* out;
  int64_t ldw, ldo;
  int N;
};

// The timesteps' cosines and sines [M, K] to LDS, as time_sinusoid_kernel forms them
template <typename TT> struct Sinusoid {
  const TT* t;
  float neg_log_period, scale, pre;
};
template <typename T, typename TT>
__device__ __forceinline__ void stage_sinusoid(const Sinusoid<TT>& a, u32x4* xs, int rows, int K, int pitch) {
  const int half = K / 2;
  T* const to = reinterpret_cast<T*>(xs);
  for (int i = threadIdx.x; i < rows * half; i += kWaves * 64) {
    const int m = i / half, j = i - m * half;
    time_sinusoid<T>(a.t[m], j, half, a.neg_log_period, a.scale, a.pre, to[m * pitch * 8 + j], to[m * pitch * 8 + half + j]);
  }
}

// tiles0: of the first weight. PAIR: of two (a template, so that one costs no selects: 442368 features, two rows 418 us, with them 421). `from`: the
// workgroup's first tile.
template <typename T, bool PAIR, typename Stage>
__device__ __forceinline__ void few_rows(Stage&& stage, const FewOut<T>& o0, const FewOut<T>& o1, int M, int K, int tiles0, int tiles, int from) {
  extern __shared__ u32x4 lds[];
  f32x4* red = reinterpret_cast<f32x4*>(lds);
  u32x4* xs = lds + kRedBytes / 16;
  const int vecs = K / 8, pitch = vecs + 1;  // 16-byte vectors of a row of x
  stage(xs, vecs, pitch);
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;
  const int steps_all = K / kStepK, per_wave = (steps_all + kWaves - 1) / kWaves;
  const int first = min(wave * per_wave, steps_all), count = min(per_wave, steps_all - first);
  const int chunks = (per_wave + kSteps - 1) / kSteps;
  const u32x4* xrow = xs + min(col, M - 1) * pitch + quad;

  // loads past the wave's share repeat its last step (an L1 hit); a wave without a share reads the row's last step
  auto fetch = [&](u32x4 (&r)[kSteps], int tile, int chunk) {
    const bool second = PAIR && tile >= tiles0;  // (uniform; past the last tile too)
    const int row = min((second ? tile - tiles0 : tile) * kTile + col, (second ? o1.N : o0.N) - 1);
    const T* p = (second ? o1.w : o0.w) + row * (second ? o1.ldw : o0.ldw) + quad * 8;
    const int last = max(first + count - 1, 0);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int step = min(min(first + chunk * kSteps + s, last), steps_all - 1);
      r[s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + step * kStepK));
    }
  };
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int turn = 0;
  auto use = [&](const u32x4 (&r)[kSteps], int tile, int chunk) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int step = chunk * kSteps + s;
      if (step < count) acc = mfma16<T>(r[s], xrow[(first + step) * (kStepK / 8)], acc);
    }
    if (chunk + 1 < chunks) return;
    f32x4* buf = red + (turn & 1) * kWaves * 64;
    buf[wave * 64 + lane] = acc;
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    if (wave == (turn & (kWaves - 1))) {
      f32x4 sum = buf[lane];
#pragma unroll
      for (int q = 1; q < kWaves; ++q) sum += buf[q * 64 + lane];
      const bool second = PAIR && tile >= tiles0;
      const int n = (second ? tile - tiles0 : tile) * kTile + quad * 4, N = second ? o1.N : o0.N;
      const T* const bias = second ? o1.bias : o0.bias;
      T* const out = (second ? o1.out : o0.out) + col * (second ? o1.ldo : o0.ldo);
      if (col < M) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) out[n + j] = from_float<T>(sum[j] + (bias != nullptr ? to_float(bias[n + j]) : 0.f));
      }
    }
    ++turn;
  };

  // Every wave of the workgroup runs the same number of chunks, so the barriers meet. The loads are never under a condition
  // (past the last tile they repeat the last row): the compiler then knows how many are younger than those it waits for.
  u32x4 a[kSteps], b[kSteps];
  auto next = [&](int& tile, int& chunk) {
    if (++chunk == chunks) { chunk = 0; tile += gridDim.x; }
  };
  int tile = from, chunk = 0;
  fetch(a, tile, chunk);
  while (true) {
    int tile1 = tile, chunk1 = chunk;
    next(tile1, chunk1);
    fetch(b, tile1, chunk1);
    use(a, tile, chunk);
    if (tile1 >= tiles) break;
    tile = tile1; chunk = chunk1;
    next(tile, chunk);
    fetch(a, tile, chunk);
    use(b, tile1, chunk1);
    if (tile >= tiles) break;
  }
}

// What a launch does where *few, on the device, is 0 (time_tokens.hip): nothing of the kind; the next product's operand for all tokens, of `vecs` 16-byte
// vectors; all tokens' rows for the first product (`out` null: nothing).
struct Always {
  __device__ __forceinline__ bool instead() const { return false; }
};
template <typename T> struct OrSilu {
  const int* few;
  const T* x;
  T* out;
  int64_t vecs;
  __device__ __forceinline__ bool instead() const {
    if (*few != 0) return false;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * (kWaves * 64);
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * (kWaves * 64) + threadIdx.x; i < vecs; i += 4 * stride) {
      u32x4 r[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j * stride < vecs) r[j] = load_raw(x + (i + j * stride) * 8);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j * stride < vecs) store_raw(out + (i + j * stride) * 8, silu8<T>(r[j]));
    }
    return true;
  }
};
template <typename T, typename TT> struct OrSinusoid {
  const int* few;
  const TT* t;
  T* out;
  int64_t items;  // tokens times `half`
  int half;
  float neg_log_period, scale;
  __device__ __forceinline__ bool instead() const {
    if (*few != 0) return false;
    if (out == nullptr) return true;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * (kWaves * 64) + threadIdx.x; i < items; i += static_cast<int64_t>(gridDim.x) * (kWaves * 64)) {
      const int64_t row = i / half;
      const int j = static_cast<int>(i - row * half);
      time_sinusoid<T>(t[row], j, half, neg_log_period, scale, 1.f, out[row * 2 * half + j], out[row * 2 * half + half + j]);
    }
    return true;
  }
};

template <typename T, bool SILU, bool PAIR, typename Or>
__global__ __launch_bounds__(kWaves * 64, 6) void linear_few_kernel(const T* __restrict__ x, const FewOut<T> o0, const FewOut<T> o1, int M, int K,
                                                                    int64_t ldx, int tiles0, int tiles, const Or other) {
  if (other.instead()) return;
  few_rows<T, PAIR>([&](u32x4* xs, int vecs, int pitch) { stage_rows<T, SILU>(x, xs, M, vecs, pitch, ldx); }, o0, o1, M, K, tiles0, tiles, blockIdx.x);
}
template <typename T, typename TT, typename Or>
__global__ __launch_bounds__(kWaves * 64, 6) void linear_few_sinusoid_kernel(const Sinusoid<TT> a, const FewOut<T> o, int M, int K, int tiles,
                                                                             const Or other) {
  if (other.instead()) return;
  few_rows<T, false>([&](u32x4* xs, int, int pitch) { stage_sinusoid<T, TT>(a, xs, M, K, pitch); }, o, o, M, K, tiles, tiles, blockIdx.x);
}

// (groups of R features; those of the first weight come first)
template <typename T, bool SILU, int M, int R, bool PAIR, typename Or>
__global__ __launch_bounds__(kWaves * 64, 6) void linear_stream_kernel(const T* __restrict__ x, const FewOut<T> o0, const FewOut<T> o1, int rows, int K,
                                                                       int64_t ldx, const Or other) {
  if (other.instead()) return;
  extern __shared__ u32x4 lds[];
  const int vecs = K / 8;
  stage_rows<T, SILU>(x, lds, rows, vecs, vecs, ldx);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int groups0 = (o0.N + R - 1) / R, groups = groups0 + (PAIR ? (o1.N + R - 1) / R : 0);
  const int chunks = K / 512, stride = gridDim.x * kWaves;
  auto fetch = [&](u32x4 (&r)[R], int g, int c) {
    const bool second = PAIR && g >= groups0;  // (uniform; past the last group too)
    const T* const mine = (second ? o1.w : o0.w) + lane * 8 + c * 512;
    const int64_t ldw = second ? o1.ldw : o0.ldw;
    const int n0 = (second ? g - groups0 : g) * R, last = (second ? o1.N : o0.N) - 1;
#pragma unroll
    for (int i = 0; i < R; ++i) r[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(mine + min(n0 + i, last) * ldw));
  };
  float acc[R][M];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[i][m] = 0.f;
  auto use = [&](const u32x4 (&r)[R], int g, int c) {
    float xv[M][8];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const u32x4 v = lds[min(m, rows - 1) * vecs + c * 64 + lane];
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[m][j] = Raw<T>::get(v, j);
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float wv = Raw<T>::get(r[i], j);
#pragma unroll
        for (int m = 0; m < M; ++m) acc[i][m] = fmaf(wv, xv[m][j], acc[i][m]);
      }
    if (c + 1 < chunks) return;
    float mine_sum = 0.f;
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const float s = wave_sum(acc[i][m]);
        if (lane == i * M + m) mine_sum = s;
        acc[i][m] = 0.f;
      }
    const bool second = PAIR && g >= groups0;
    const int n = (second ? g - groups0 : g) * R + lane / M, m = lane % M;
    const T* const bias = second ? o1.bias : o0.bias;
    T* const out = second ? o1.out : o0.out;
    if (lane < R * M && n < (second ? o1.N : o0.N) && m < rows)
      out[m * (second ? o1.ldo : o0.ldo) + n] = from_float<T>(mine_sum + (bias != nullptr ? to_float(bias[n]) : 0.f));
  };
  u32x4 a[R], b[R];
  auto next = [&](int& g, int& c) {
    if (++c == chunks) { c = 0; g += stride; }
  };
  int g = blockIdx.x * kWaves + wave, c = 0;
  if (g >= groups) return;
  fetch(a, g, c);
  while (true) {  // (past the last group the loads repeat the last row)
    int g1 = g, c1 = c;
    next(g1, c1);
    fetch(b, g1, c1);
    use(a, g, c);
    if (g1 >= groups) break;
    g = g1; c = c1;
    next(g, c);
    fetch(a, g, c);
    use(b, g1, c1);
    if (g >= groups) break;
  }
}

// Up to three embedders, two projections each with a SiLU between, and the sum of their results. Each by itself is a chain of two launches that wait
// more than they read (2 to 5 and 19 MB at width 3072), and none hangs on another: the first projections are one launch, the second ones and the sums
// another, in which the wavefronts of a workgroup share out the embedders of the features and meet in LDS. Timestep, guidance and 768 values of pooled
// text at width 3072, one row, us under the profiler: 5.7 + 7.7, 5.8 + 7.4, 5.4 + 7.4 and two sums of 4.8 / 9.3 + 13.5; a step of 1024 + 512 tokens without
// it 4455 -> 4434.
constexpr int kEmbedders = 3;
struct EmbedInput {
  const void* x;  // timesteps [M], or rows
  int64_t ldx;
  int K, t_dtype;  // t_dtype -1: rows
  float neg_log_period, scale, pre;
};
template <typename T> struct EmbedFirst {
  EmbedInput in[kEmbedders];
  FewOut<T> out[kEmbedders];
};
template <typename T>
__global__ __launch_bounds__(kWaves * 64, 6) void embed_first_kernel(const EmbedFirst<T> p, int M, int tiles) {
  const int which = blockIdx.x / tiles;
  const EmbedInput& in = p.in[which];
  few_rows<T, false>([&](u32x4* xs, int vecs, int pitch) {
    auto sinusoid = [&](auto type) {
      using TT = decltype(type);
      stage_sinusoid<T, TT>(Sinusoid<TT>{static_cast<const TT*>(in.x), in.neg_log_period, in.scale, in.pre}, xs, M, in.K, pitch);
    };
    if (in.t_dtype < 0) stage_rows<T, false>(static_cast<const T*>(in.x), xs, M, vecs, pitch, in.ldx);
    else if (in.t_dtype == ODIT_F32) sinusoid(0.f);
    else if (in.t_dtype == ODIT_BF16) sinusoid(bf16_t{});
    else sinusoid(f16_t{});
  }, p.out[which], p.out[which], M, in.K, tiles, tiles, static_cast<int>(blockIdx.x) - which * tiles);
}

template <typename T> struct EmbedSecond {
  const T* hidden;  // [count, rows, N]
  const T *w[kEmbedders], *bias[kEmbedders];
  int64_t ldw[kEmbedders];
  T* out;
};
template <typename T, int M>
__global__ __launch_bounds__(kWaves * 64, 6) void embed_second_kernel(const EmbedSecond<T> p, int count, int rows, int N) {
  constexpr int R = 2;  // features of a wavefront
  extern __shared__ u32x4 lds[];
  __shared__ float part[kWaves][R * M];
  const int vecs = N / 8, each = rows * vecs;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int places = kWaves / count, which = wave % count, place = wave / count;
  const int g = blockIdx.x * places + place, chunks = N / 512;
  const T* const mine = p.w[which] + lane * 8;
  auto fetch = [&](u32x4 (&r)[R], int c) {  // (past the last feature and the last chunk the loads repeat it)
#pragma unroll
    for (int i = 0; i < R; ++i)
      r[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(mine + min(g * R + i, N - 1) * p.ldw[which] + min(c, chunks - 1) * 512));
  };
  u32x4 a[R], b[R];
  fetch(a, 0);
  stage_rows<T, true>(p.hidden, lds, count * rows, vecs, vecs, N);
  __syncthreads();
  if (place < places && g * R < N) {
    const u32x4* const x = lds + which * each + lane;
    float acc[R][M];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int m = 0; m < M; ++m) acc[i][m] = 0.f;
    auto use = [&](const u32x4 (&r)[R], int c) {  // (linear_stream_kernel's sums)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const u32x4 v = x[min(m, rows - 1) * vecs + c * 64];
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[i][m] = fmaf(Raw<T>::get(r[i], j), Raw<T>::get(v, j), acc[i][m]);
      }
    };
    for (int c = 0;;) {
      fetch(b, c + 1);
      use(a, c);
      if (++c >= chunks) break;
      fetch(a, c + 1);
      use(b, c);
      if (++c >= chunks) break;
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const float s = wave_sum(acc[i][m]);
        const T* const bias = p.bias[which];
        if (lane == i * M + m)
          part[wave][lane] = to_float(from_float<T>(s + (bias != nullptr ? to_float(bias[min(g * R + i, N - 1)]) : 0.f)));
      }
  }
  __syncthreads();
  if (threadIdx.x < places * R * M) {
    const int at = threadIdx.x / (R * M), i = threadIdx.x % (R * M) / M, m = threadIdx.x % M, n = (blockIdx.x * places + at) * R + i;
    if (n < N && m < rows) {
      float v = part[at * count][i * M + m];
      for (int e = 1; e < count; ++e) v = to_float(from_float<T>(v + part[at * count + e][i * M + m]));
      p.out[static_cast<int64_t>(m) * N + n] = from_float<T>(v);
    }
  }
}

// Rows of W a wavefront takes at a time: two; four (twice the loads in flight, half the steps) where every wavefront of the grid
// has three or more such groups and one or two rows of x leave the registers for it: N=442368, two rows of x 414 / 405 us,
// 73728 69.5 / 68.1, but 36864 36.5 / 37.3, 9216 13.2 / 15.0; with four rows of x 440 / 566.
constexpr int kStreamWide = 1 << 16;

template <typename T, bool SILU, bool PAIR, typename Or>
int launch_stream(const T* x, const FewOut<T>& o0, const FewOut<T>& o1, int M, int K, int64_t ldx, int slots, const Or& other, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(M) * K * 2;
  const int N = o0.N + (PAIR ? o1.N : 0);
#define ODIT_STREAM(ROWS, R)                                                                                                             \
  do {                                                                                                                                   \
    const int groups = (o0.N + R - 1) / R + (PAIR ? (o1.N + R - 1) / R : 0), wanted = (groups + kWaves - 1) / kWaves;                      \
    linear_stream_kernel<T, SILU, ROWS, R, PAIR, Or><<<wanted < slots ? wanted : slots, kWaves * 64, lds, stream>>>(x, o0, o1, M, K, ldx, other); \
  } while (0)
  if constexpr (!std::is_same<Or, Always>::value) {
    // four rows; every place on the chip, for what the launch may do instead (5120 features alone would be 320 workgroups, two on some compute units)
    linear_stream_kernel<T, SILU, 4, 2, PAIR, Or><<<slots, kWaves * 64, lds, stream>>>(x, o0, o1, M, K, ldx, other);
    return check_launch("odit_linear_few (stream)");
  }
  if (M > 2) ODIT_STREAM(4, 2);
  else if (N >= kStreamWide && M == 2) ODIT_STREAM(2, 4);
  else if (N >= kStreamWide) ODIT_STREAM(1, 4);
  else if (M == 2) ODIT_STREAM(2, 2);
  else ODIT_STREAM(1, 2);
#undef ODIT_STREAM
  return check_launch("odit_linear_few (stream)");
}

// Taken: up to 16 rows of x (the columns of one MFMA operand) that fit a CU's LDS; three workgroups per CU while they fit,
// one still has 64 KB of loads in flight.
constexpr int kFewMaxRows = 16, kFewMaxGroups = 3, kStreamMaxRows = 4;
constexpr size_t kFewMaxLds = 160 * 1024;

// whether a reduction is the stream kernel's
bool few_streams(int M, int K) { return M <= kStreamMaxRows && K % 512 == 0 && static_cast<size_t>(M) * K * 2 <= kFewMaxLds / kFewMaxGroups; }

size_t few_lds(int M, int K) { return kRedBytes + static_cast<size_t>(M) * (K / 8 + 1) * 16; }
int few_grid(int tiles, size_t lds, int cus) {
  const int fit = static_cast<int>(kFewMaxLds / lds), slots = cus * (fit < kFewMaxGroups ? fit : kFewMaxGroups);
  return tiles < slots ? tiles : slots;
}

struct FewArgs { const void *w, *bias; void* out; int N; int64_t ldw, ldo; };

// How many rows a wavefront takes at a time follows from the features
// of both; the bits do not (a feature's sum is one wavefront's).
template <typename T, bool SILU, bool PAIR, typename Or = Always>
int run_few(const void* x, const FewArgs* a, int M, int K, int64_t ldx, int cus, hipStream_t stream, const Or& other = Or{}) {
  FewOut<T> o[2];
  for (int i = 0; i < 2; ++i)  // (without a second weight nothing reads the second)
    o[i] = FewOut<T>{static_cast<const T*>(a[i].w), static_cast<const T*>(a[i].bias), static_cast<T*>(a[i].out), a[i].ldw, a[i].ldo, a[i].N};
  if (few_streams(M, K))
    return launch_stream<T, SILU, PAIR>(static_cast<const T*>(x), o[0], o[1], M, K, ldx, cus * kFewMaxGroups, other, stream);
  const int tiles0 = (a[0].N + kTile - 1) / kTile, tiles = tiles0 + (PAIR ? (a[1].N + kTile - 1) / kTile : 0);
  const size_t lds = few_lds(M, K);
  linear_few_kernel<T, SILU, PAIR, Or><<<few_grid(tiles, lds, cus), kWaves * 64, lds, stream>>>(static_cast<const T*>(x), o[0], o[1], M, K, ldx, tiles0, tiles,
                                                                                                other);
  return check_launch("odit_linear_few");
}

template <typename T, typename TT, typename Or = Always>
int run_sinusoid(const void* t, float neg_log_period, float scale, float pre, const FewArgs& a, int M, int K, int cus, hipStream_t stream,
                 const Or& other = Or{}) {
  const FewOut<T> o{static_cast<const T*>(a.w), static_cast<const T*>(a.bias), static_cast<T*>(a.out), a.ldw, a.ldo, a.N};
  const int tiles = (a.N + kTile - 1) / kTile;
  const size_t lds = few_lds(M, K);
  linear_few_sinusoid_kernel<T, TT, Or><<<few_grid(tiles, lds, cus), kWaves * 64, lds, stream>>>(
      Sinusoid<TT>{static_cast<const TT*>(t), neg_log_period, scale, pre}, o, M, K, tiles, other);
  return check_launch("odit_time_linear");
}

template <typename T>
int run_embed(const odit_embedder* e, int count, int M, int N, void* hidden, void* out, hipStream_t stream) {
  EmbedFirst<T> a;
  EmbedSecond<T> b;
  int widest = 0;
  b.hidden = static_cast<const T*>(hidden);
  b.out = static_cast<T*>(out);
  for (int i = 0; i < kEmbedders; ++i) {
    const odit_embedder& m = e[i < count ? i : 0];
    a.in[i] = EmbedInput{m.x, m.ldx, m.K, m.t_dtype, m.neg_log_period, m.scale, m.pre};
    a.out[i] = FewOut<T>{static_cast<const T*>(m.w1), static_cast<const T*>(m.bias1), static_cast<T*>(hidden) + static_cast<int64_t>(i) * M * N, m.ldw1, N, N};
    b.w[i] = static_cast<const T*>(m.w2);
    b.bias[i] = static_cast<const T*>(m.bias2);
    b.ldw[i] = m.ldw2;
    if (m.K > widest) widest = m.K;
  }
  const int tiles = (N + kTile - 1) / kTile;
  embed_first_kernel<T><<<count * tiles, kWaves * 64, few_lds(M, widest), stream>>>(a, M, tiles);
  const int rc = check_launch("odit_embed_sum");
  if (rc != ODIT_OK) return rc;
  const int groups = (N + 1) / 2, places = kWaves / count;
  const dim3 grid((groups + places - 1) / places);
  const size_t lds = static_cast<size_t>(count) * M * N * 2;
  if (M > 2) embed_second_kernel<T, 4><<<grid, kWaves * 64, lds, stream>>>(b, count, M, N);
  else if (M == 2) embed_second_kernel<T, 2><<<grid, kWaves * 64, lds, stream>>>(b, count, M, N);
  else embed_second_kernel<T, 1><<<grid, kWaves * 64, lds, stream>>>(b, count, M, N);
  return check_launch("odit_embed_sum");
}

}  // namespace
}  // namespace odit

static int few_check(const char* name, const odit::FewArgs* a, int count, int M, int K, int dtype) {
  using namespace odit;
  ODIT_CHECK_ARG(M >= 0 && K > 0, "%s: bad shape M=%d K=%d", name, M, K);
  const size_t lds = few_lds(M, K);
  bool takes = (dtype == ODIT_BF16 || dtype == ODIT_F16) && M <= kFewMaxRows && K % kStepK == 0 && lds <= kFewMaxLds;
  for (int i = 0; i < count; ++i) {
    ODIT_CHECK_ARG(a[i].w && a[i].out, "%s: w/out must not be null", name);
    ODIT_CHECK_ARG(a[i].N > 0, "%s: bad shape N=%d", name, a[i].N);
    ODIT_CHECK_ARG(a[i].ldw >= K && a[i].ldo >= a[i].N, "%s: leading dimensions too small", name);
    takes = takes && a[i].ldw % 8 == 0 && aligned16(a[i].w);
  }
  if (!takes) {
    set_error("%s: takes 16-bit types, M <= %d, K a multiple of %d, 16-byte aligned rows and M (K + 8) 2 bytes of LDS (M=%d N=%d K=%d)", name, kFewMaxRows,
              kStepK, M, a[0].N, K);
    return ODIT_ENOTSUP;
  }
  return ODIT_OK;
}

static int few_go(const char* name, const void* x, odit::FewArgs (&a)[2], int count, int M, int K, int64_t ldx, int dtype, int silu_input, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(x != nullptr, "%s: x must not be null", name);
  ODIT_CHECK_ARG(ldx >= K, "%s: leading dimensions too small", name);
  const int rc = few_check(name, a, count, M, K, dtype);
  if (rc != ODIT_OK) return rc;
  if (ldx % 8 != 0 || !aligned16(x)) { set_error("%s: rows of x must be 16-byte aligned", name); return ODIT_ENOTSUP; }
  if (M == 0) return ODIT_OK;
  const int cus = device_cus();
  if (cus <= 0) { set_error("%s: cannot read the device's compute-unit count", name); return ODIT_ELAUNCH; }
  const hipStream_t s = static_cast<hipStream_t>(stream);
#define ODIT_FEW(T, SILU) (count == 2 ? run_few<T, SILU, true>(x, a, M, K, ldx, cus, s) : run_few<T, SILU, false>(x, a, M, K, ldx, cus, s))
  if (dtype == ODIT_BF16) return silu_input ? ODIT_FEW(bf16_t, true) : ODIT_FEW(bf16_t, false);
  return silu_input ? ODIT_FEW(f16_t, true) : ODIT_FEW(f16_t, false);
#undef ODIT_FEW
}

int odit::linear_few_or(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int dtype, const FewOr& other, bool ask,
                        hipStream_t stream) {
  const FewArgs a[2] = {{w, bias, out, N, ldw, N}, {}};
  const int rc = few_check("odit_linear_few", a, 1, M, K, dtype);
  if (rc != ODIT_OK || ask) return rc;
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear_few: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
#define ODIT_OR(T) \
  run_few<T, true, false>(x, a, M, K, K, cus, stream, OrSilu<T>{other.few, static_cast<const T*>(other.x), static_cast<T*>(other.out), other.n})
  return dtype == ODIT_BF16 ? ODIT_OR(bf16_t) : ODIT_OR(f16_t);
#undef ODIT_OR
}

int odit::time_linear_or(const void* t, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, float neg_log_period, float scale,
                         int t_dtype, int dtype, const FewOr& other, bool ask, hipStream_t stream) {
  const FewArgs a{w, bias, out, N, ldw, N};
  const int rc = few_check("odit_time_linear", &a, 1, M, K, dtype);
  if (rc != ODIT_OK || ask) return rc;
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_time_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
#define ODIT_OR(T)                                                                                                                       \
  run_sinusoid<T, TT>(t, neg_log_period, scale, 1.f, a, M, K, cus, stream,                                                                \
                      OrSinusoid<T, TT>{other.few, static_cast<const TT*>(other.x), static_cast<T*>(other.out), other.n * (K / 2), K / 2, \
                                        neg_log_period, scale})
  ODIT_DISPATCH_DTYPE(t_dtype, TT, { return dtype == ODIT_BF16 ? ODIT_OR(bf16_t) : ODIT_OR(f16_t); });
#undef ODIT_OR
  return ODIT_OK;
}

extern "C" int odit_linear_few(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldx,
                               int64_t ldw, int64_t ldo, int dtype, int silu_input, void* stream) {
  odit::FewArgs a[2] = {{w, bias, out, N, ldw, ldo}, {}};
  return few_go("odit_linear_few", x, a, 1, M, K, ldx, dtype, silu_input, stream);
}

extern "C" int odit_linear_few_pair(const void* x, const void* const w[2], const void* const bias[2], void* const out[2], int M, const int N[2], int K,
                                    int64_t ldx, const int64_t ldw[2], const int64_t ldo[2], int dtype, int silu_input, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(w && bias && out && N && ldw && ldo, "odit_linear_few_pair: null arguments");
  FewArgs a[2];
  for (int i = 0; i < 2; ++i) a[i] = FewArgs{w[i], bias[i], out[i], N[i], ldw[i], ldo[i]};
  ODIT_CHECK_ARG(static_cast<int64_t>(N[0]) + N[1] < (1ll << 31) - 64, "odit_linear_few_pair: too many features");
  return few_go("odit_linear_few_pair", x, a, 2, M, K, ldx, dtype, silu_input, stream);
}

extern "C" int odit_time_linear(const void* t, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int64_t ldo,
                                float neg_log_period, float scale, float pre, int t_dtype, int dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(t != nullptr, "odit_time_linear: t must not be null");
  const FewArgs a{w, bias, out, N, ldw, ldo};
  const int rc = few_check("odit_time_linear", &a, 1, M, K, dtype);
  if (rc != ODIT_OK) return rc;
  // (a reduction that the stream kernel would take has another order of summation)
  if (few_streams(M, K)) {
    set_error("odit_time_linear: K=%d is the stream kernel's", K);
    return ODIT_ENOTSUP;
  }
  if (M == 0) return ODIT_OK;
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_time_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const hipStream_t s = static_cast<hipStream_t>(stream);
  ODIT_DISPATCH_DTYPE(t_dtype, TT, {
    return dtype == ODIT_BF16 ? run_sinusoid<bf16_t, TT>(t, neg_log_period, scale, pre, a, M, K, cus, s)
                              : run_sinusoid<f16_t, TT>(t, neg_log_period, scale, pre, a, M, K, cus, s);
  });
  return ODIT_OK;
}

extern "C" int odit_embed_sum(const odit_embedder* embedders, int count, int M, int N, void* hidden, void* out, int dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(embedders && hidden && out, "odit_embed_sum: null arguments");
  ODIT_CHECK_ARG(count >= 1 && count <= kEmbedders && M >= 0 && N > 0, "odit_embed_sum: bad shape count=%d M=%d N=%d", count, M, N);
  bool takes = N % 8 == 0 && aligned16(hidden) && few_streams(M, N) && static_cast<size_t>(count) * M * N * 2 <= kFewMaxLds - kWaves * 64;
  for (int i = 0; i < count; ++i) {
    const odit_embedder& e = embedders[i];
    ODIT_CHECK_ARG(e.x && e.K > 0, "odit_embed_sum: bad input of embedder %d", i);
    ODIT_CHECK_ARG(e.t_dtype >= -1 && e.t_dtype <= ODIT_F32, "odit_embed_sum: bad timestep type %d", e.t_dtype);
    const FewArgs a[2] = {{e.w1, e.bias1, hidden, N, e.ldw1, N}, {e.w2, e.bias2, out, N, e.ldw2, N}};
    int rc = few_check("odit_embed_sum", a, 1, M, e.K, dtype);
    if (rc == ODIT_OK) rc = few_check("odit_embed_sum", a + 1, 1, M, N, dtype);
    if (rc != ODIT_OK) return rc;
    // (a first projection that the stream kernel would take has another order of summation)
    takes = takes && !few_streams(M, e.K) && (e.t_dtype < 0 ? e.ldx >= e.K && e.ldx % 8 == 0 && aligned16(e.x) : e.K % 2 == 0);
  }
  if (!takes) {
    set_error("odit_embed_sum: takes up to %d rows, N a multiple of 512, rows of 16-byte alignment and first reductions that odit_linear_few's matrix kernel runs "
              "(count=%d M=%d N=%d)", kStreamMaxRows, count, M, N);
    return ODIT_ENOTSUP;
  }
  if (M == 0) return ODIT_OK;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == ODIT_BF16 ? run_embed<bf16_t>(embedders, count, M, N, hidden, out, s) : run_embed<f16_t>(embedders, count, M, N, hidden, out, s);
}
