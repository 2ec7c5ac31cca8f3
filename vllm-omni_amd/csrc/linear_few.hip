// Projections of a few rows (M <= 16): the timestep embedding, the modulation parameters of all blocks from one stacked
// weight, the head's norm. out[M,N] = act(x)[M,K] W[N,K]^T + bias, act = identity or SiLU rounded to the tensor type.
//
// Bound: the weights are read once (N K 2 bytes: 453 MB for two blocks of width 3072) and everything else is noise, so
// the kernel is a weight stream with enough loads in flight: 8 to 12 KB per wave, 24 waves per CU. From cold caches, against
// the library's first choice: N=73728, K=3072, two rows 176 -> 93 us (4.9 TB/s; a large copy reaches 4.95); N=36864 95 -> 51;
// N=30720, K=5120 114 -> 75; N=3072, K=3072 20 -> 11; N=3072, K=256 11 -> 7.6. Loads are non-temporal: without, the weights
// push activations out of the last-level cache and wait for their write-back (N=73728: 141 us). kSteps of 6 or 12 measured
// the same at K=3072 and 15 % slower at K=5120, whose 20 steps per wave they do not divide.
//
// A workgroup of 8 waves takes 16 features at a time; the waves divide the reduction. A wave loads 16 features x 32
// reduction elements with one 16-byte load per lane, straight into the A operand of v_mfma_f32_16x16x32 (lane l: feature
// l % 16, elements 8 (l / 16) ..); adjacent loads of a wave cover the rest of the lines. kSteps loads are in flight while the
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

template <typename T, bool SILU>
__global__ __launch_bounds__(kWaves * 64, 6) void linear_few_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                                    const T* __restrict__ bias, T* __restrict__ out, int M,
                                                                    int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                                                    int tiles) {
  extern __shared__ u32x4 lds[];
  f32x4* red = reinterpret_cast<f32x4*>(lds);
  u32x4* xs = lds + kRedBytes / 16;
  const int vecs = K / 8, pitch = vecs + 1;  // 16-byte vectors of a row of x
  for (int i = threadIdx.x; i < M * vecs; i += kWaves * 64) {
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

template <typename T, bool SILU>
int launch_few(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldx, int64_t ldw,
               int64_t ldo, int grid, int tiles, size_t lds, hipStream_t stream) {
  linear_few_kernel<T, SILU><<<grid, kWaves * 64, lds, stream>>>(static_cast<const T*>(x), static_cast<const T*>(w),
                                                                 static_cast<const T*>(bias), static_cast<T*>(out), M, N, K,
                                                                 ldx, ldw, ldo, tiles);
  return check_launch("odit_linear_few");
}

}  // namespace
}  // namespace odit

// Taken: up to 16 rows of x (the columns of one MFMA operand) that fit a CU's LDS; three workgroups per CU while they fit,
// one still has 64 KB of loads in flight.
constexpr int kFewMaxRows = 16, kFewMaxGroups = 3;
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
  if (dtype == ODIT_BF16)
    return silu_input ? launch_few<bf16_t, true>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s)
                      : launch_few<bf16_t, false>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s);
  return silu_input ? launch_few<f16_t, true>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s)
                    : launch_few<f16_t, false>(x, w, bias, out, M, N, K, ldx, ldw, ldo, grid, tiles, lds, s);
}
