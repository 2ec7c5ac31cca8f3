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
#include "odit_common.h"
#include "gemm_bf16.h"

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

// x, activated, to LDS: `rows` rows of `vecs` 16-byte vectors, `pitch` apart
template <typename T, bool SILU>
__device__ __forceinline__ void stage_rows(const T* __restrict__ x, u32x4* xs, int rows, int vecs, int pitch, int64_t ldx) {
  for (int i = threadIdx.x; i < rows * vecs; i += kWaves * 64) {
    const int m = i / vecs, v = i - m * vecs;
    u32x4 r = load_raw(x + m * ldx + v * 8);
    if (SILU) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const float a = Raw<T>::get(r, 2 * p), b = Raw<T>::get(r, 2 * p + 1);
        Raw<T>::set2(r, p, a / (1.f + __expf(-a)), b / (1.f + __expf(-b)));
      }
    }
    xs[m * pitch + v] = r;
  }
}

template <typename T, bool SILU>
__global__ __launch_bounds__(kWaves * 64, 6) void linear_few_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                                    const T* __restrict__ bias, T* __restrict__ out, int M,
                                                                    int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                                                    int tiles) {
  extern __shared__ u32x4 lds[];
  f32x4* red = reinterpret_cast<f32x4*>(lds);
  u32x4* xs = lds + kRedBytes / 16;
  const int vecs = K / 8, pitch = vecs + 1;  // 16-byte vectors of a row of x
  stage_rows<T, SILU>(x, xs, M, vecs, pitch, ldx);
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;
  const int steps_all = K / kStepK, per_wave = (steps_all + kWaves - 1) / kWaves;
  const int first = min(wave * per_wave, steps_all), count = min(per_wave, steps_all - first);
  const int chunks = (per_wave + kSteps - 1) / kSteps;
  const u32x4* xrow = xs + min(col, M - 1) * pitch + quad;

  // loads past the wave's share repeat its last step (an L1 hit); a wave without a share reads the row's last step
  auto fetch = [&](u32x4 (&r)[kSteps], int tile, int chunk) {
    const T* p = w + static_cast<int64_t>(min(tile * kTile + col, N - 1)) * ldw + quad * 8;
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
      const int n = tile * kTile + quad * 4;
      if (col < M) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) out[col * ldo + n + j] = from_float<T>(sum[j] + (bias != nullptr ? to_float(bias[n + j]) : 0.f));
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
  int tile = blockIdx.x, chunk = 0;
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

template <typename T, bool SILU, int M, int R>
__global__ __launch_bounds__(kWaves * 64, 6) void linear_stream_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                                       const T* __restrict__ bias, T* __restrict__ out, int rows,
                                                                       int N, int K, int64_t ldx, int64_t ldw, int64_t ldo) {
  extern __shared__ u32x4 lds[];
  const int vecs = K / 8;
  stage_rows<T, SILU>(x, lds, rows, vecs, vecs, ldx);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunks = K / 512, groups = (N + R - 1) / R, stride = gridDim.x * kWaves;
  const T* const mine = w + lane * 8;
  auto fetch = [&](u32x4 (&r)[R], int g, int c) {
#pragma unroll
    for (int i = 0; i < R; ++i)
      r[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(mine + static_cast<int64_t>(min(g * R + i, N - 1)) * ldw + c * 512));
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
    const int n = g * R + lane / M, m = lane % M;
    if (lane < R * M && n < N && m < rows) out[m * ldo + n] = from_float<T>(mine_sum + (bias != nullptr ? to_float(bias[n]) : 0.f));
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

template <typename T, bool SILU>
int launch_few(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldx, int64_t ldw,
               int64_t ldo, int grid, int tiles, size_t lds, hipStream_t stream) {
  linear_few_kernel<T, SILU><<<grid, kWaves * 64, lds, stream>>>(static_cast<const T*>(x), static_cast<const T*>(w),
                                                                 static_cast<const T*>(bias), static_cast<T*>(out), M, N, K,
                                                                 ldx, ldw, ldo, tiles);
  return check_launch("odit_linear_few");
}

// Rows of W a wavefront takes at a time: two; four (twice the loads in flight, half the steps) where every wavefront of the grid
// has three or more such groups and one or two rows of x leave the registers for it: N=442368, two rows of x 414 / 405 us,
// 73728 69.5 / 68.1, but 36864 36.5 / 37.3, 9216 13.2 / 15.0; with four rows of x 440 / 566.
constexpr int kStreamWide = 1 << 16;

template <typename T, bool SILU>
int launch_stream(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int slots,
                  hipStream_t stream) {
  const size_t lds = static_cast<size_t>(M) * K * 2;
#define ODIT_STREAM(ROWS, R)                                                                                                             \
  do {                                                                                                                                   \
    const int wanted = (N + R * kWaves - 1) / (R * kWaves);                                                                              \
    linear_stream_kernel<T, SILU, ROWS, R><<<wanted < slots ? wanted : slots, kWaves * 64, lds, stream>>>(                                 \
        static_cast<const T*>(x), static_cast<const T*>(w), static_cast<const T*>(bias), static_cast<T*>(out), M, N, K, ldx, ldw, ldo);     \
  } while (0)
  if (M > 2) ODIT_STREAM(4, 2);
  else if (N >= kStreamWide && M == 2) ODIT_STREAM(2, 4);
  else if (N >= kStreamWide) ODIT_STREAM(1, 4);
  else if (M == 2) ODIT_STREAM(2, 2);
  else ODIT_STREAM(1, 2);
#undef ODIT_STREAM
  return check_launch("odit_linear_few (stream)");
}

}  // namespace
}  // namespace odit

// Taken: up to 16 rows of x (the columns of one MFMA operand) that fit a CU's LDS; three workgroups per CU while they fit,
// one still has 64 KB of loads in flight.
constexpr int kFewMaxRows = 16, kFewMaxGroups = 3, kStreamMaxRows = 4;
constexpr size_t kFewMaxLds = 160 * 1024;

extern "C" int odit_linear_few(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldx,
                               int64_t ldw, int64_t ldo, int dtype, int silu_input, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(x && w && out, "odit_linear_few: x/w/out must not be null");
  ODIT_CHECK_ARG(M >= 0 && N > 0 && K > 0, "odit_linear_few: bad shape M=%d N=%d K=%d", M, N, K);
  ODIT_CHECK_ARG(ldx >= K && ldw >= K && ldo >= N, "odit_linear_few: leading dimensions too small");
  const size_t lds = kRedBytes + static_cast<size_t>(M) * (K / 8 + 1) * 16;
  if ((dtype != ODIT_BF16 && dtype != ODIT_F16) || M > kFewMaxRows || K % kStepK != 0 || ldx % 8 != 0 || ldw % 8 != 0 ||
      !aligned16(x) || !aligned16(w) || lds > kFewMaxLds) {
    set_error("odit_linear_few: takes 16-bit types, M <= %d, K a multiple of %d, 16-byte aligned rows and M (K + 8) 2 bytes of LDS (M=%d N=%d K=%d)",
              kFewMaxRows, kStepK, M, N, K);
    return ODIT_ENOTSUP;
  }
  if (M == 0) return ODIT_OK;
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear_few: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const int tiles = (N + kTile - 1) / kTile, fit = static_cast<int>(kFewMaxLds / lds);
  const int slots = cus * (fit < kFewMaxGroups ? fit : kFewMaxGroups), grid = tiles < slots ? tiles : slots;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t stream_lds = static_cast<size_t>(M) * K * 2;
  if (M <= kStreamMaxRows && K % 512 == 0 && stream_lds <= kFewMaxLds / kFewMaxGroups) {
    const int all = cus * kFewMaxGroups;
    if (dtype == ODIT_BF16)
      return silu_input ? launch_stream<bf16_t, true>(x, w, bias, out, M, N, K, ldx, ldw, ldo, all, s)
                        : launch_stream<bf16_t, false>(x, w, bias, out, M, N, K, ldx, ldw, ldo, all, s);
    return silu_input ? launch_stream<f16_t, true>(x, w, bias, out, M, N, K, ldx, ldw, ldo, all, s)
                      : launch_stream<f16_t, false>(x, w, bias, out, M, N, K, ldx, ldw, ldo, all, s);
  }
  if (dtype == ODIT_BF16)
    return silu_input ? launch_few<bf16_t, true>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s)
                      : launch_few<bf16_t, false>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s);
  return silu_input ? launch_few<f16_t, true>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s)
                    : launch_few<f16_t, false>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s);
}
