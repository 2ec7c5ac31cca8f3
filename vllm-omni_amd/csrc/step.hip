// The small work around the transformer in a denoise step: the timestep sinusoid, the CFG combination and the Euler update.
// Every tensor here is a few KB to a few MB, so what bounds it is the number of launches and the host time of each: as torch
// operations the three were 10, 7 and 5 launches (about 2 us each on the GPU and 4 to 8 us on the host); here each is one.
// Every intermediate is rounded where the torch expression rounds it, with no contraction of multiply and add.
#include "odit_common.h"

#pragma clang fp contract(off)

namespace odit {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxBlocks = 4096;

// out[i, :] = cos | sin of scale * (t[i] * exp(-log(max_period) j / half)); the accurate exp, cos and sin, which torch calls
template <typename TT, typename T>
__global__ __launch_bounds__(kBlock) void time_sinusoid_kernel(const TT* __restrict__ t, T* __restrict__ out, int64_t n, int half,
                                                               float neg_log_period, float scale) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n * half; i += static_cast<int64_t>(gridDim.x) * kBlock) {
    const int64_t row = i / half;
    const int j = static_cast<int>(i - row * half);
    const float freq = expf(neg_log_period * static_cast<float>(j) / static_cast<float>(half));
    const float arg = scale * (to_float(t[row]) * freq);
    out[row * 2 * half + j] = from_float<T>(cosf(arg));
    out[row * 2 * half + half + j] = from_float<T>(sinf(arg));
  }
}

template <typename T> __device__ __forceinline__ float combine(float pos, float neg, float scale) {
  return round_to<T>(neg + round_to<T>(scale * round_to<T>(pos - neg)));
}

template <typename T>
__global__ __launch_bounds__(kBlock) void cfg_combine_kernel(const T* __restrict__ pos, const T* __restrict__ neg,
                                                             T* __restrict__ out, int64_t n, float scale) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * kBlock)
    out[i] = from_float<T>(combine<T>(to_float(pos[i]), to_float(neg[i]), scale));
}

// with the norm of every row (channels of a token) put back to that of the positive branch; 8 lanes per row
constexpr int kRowLanes = 8;
template <typename T>
__global__ __launch_bounds__(kBlock) void cfg_combine_norm_kernel(const T* __restrict__ pos, const T* __restrict__ neg,
                                                                  T* __restrict__ out, int64_t rows, int C, float scale) {
  const int sub = threadIdx.x % kRowLanes;
  constexpr int kRows = kBlock / kRowLanes;
  for (int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRows; row0 < rows; row0 += static_cast<int64_t>(gridDim.x) * kRows) {
    const int64_t row = row0 + threadIdx.x / kRowLanes;
    const bool live = row < rows;
    const T *p = pos + (live ? row : 0) * C, *q = neg + (live ? row : 0) * C;
    float sp = 0.f, sc = 0.f;
    for (int c = sub * 8; c < C; c += kRowLanes * 8) {
      const u32x4 a = load_raw(p + c), b = load_raw(q + c);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = Raw<T>::get(a, j), y = combine<T>(x, Raw<T>::get(b, j), scale);
        sp += x * x;
        sc += y * y;
      }
    }
    sp = row_group_sum<kRowLanes>(sp);
    sc = row_group_sum<kRowLanes>(sc);
    const float ratio = round_to<T>(round_to<T>(sqrtf(sp)) / round_to<T>(sqrtf(sc)));
    if (!live) continue;
    for (int c = sub * 8; c < C; c += kRowLanes * 8) {
      const u32x4 a = load_raw(p + c), b = load_raw(q + c);
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        Raw<T>::set2(o, j, combine<T>(Raw<T>::get(a, 2 * j), Raw<T>::get(b, 2 * j), scale) * ratio,
                     combine<T>(Raw<T>::get(a, 2 * j + 1), Raw<T>::get(b, 2 * j + 1), scale) * ratio);
      store_raw(out + row * C + c, o);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void euler_step_kernel(const T* __restrict__ x, const T* __restrict__ v, T* __restrict__ out,
                                                            int64_t n, float dt) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * kBlock)
    out[i] = from_float<T>(to_float(x[i]) + dt * to_float(v[i]));
}

int blocks_for(int64_t threads) {
  const int64_t b = (threads + kBlock - 1) / kBlock;
  return static_cast<int>(b < kMaxBlocks ? b : kMaxBlocks);
}

template <typename TT, typename T>
int launch_sinusoid(const void* t, void* out, int64_t n, int half, float neg_log_period, float scale, hipStream_t s) {
  time_sinusoid_kernel<TT, T><<<blocks_for(n * half), kBlock, 0, s>>>(static_cast<const TT*>(t), static_cast<T*>(out), n, half,
                                                                     neg_log_period, scale);
  return check_launch("odit_time_sinusoid");
}

}  // namespace
}  // namespace odit

extern "C" int odit_time_sinusoid(const void* t, void* out, int64_t n, int dim, float neg_log_period, float scale, int t_dtype,
                                  int out_dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(t && out && n >= 0 && dim > 0 && dim % 2 == 0, "odit_time_sinusoid: needs t, out and an even dim (n=%lld dim=%d)",
                 static_cast<long long>(n), dim);
  if (n == 0) return ODIT_OK;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  ODIT_DISPATCH_DTYPE(t_dtype, TT, {
    ODIT_DISPATCH_DTYPE(out_dtype, T, { return launch_sinusoid<TT, T>(t, out, n, dim / 2, neg_log_period, scale, s); });
  });
  return ODIT_OK;
}

extern "C" int odit_cfg_combine(const void* pos, const void* neg, void* out, int64_t rows, int C, float scale, int normalize,
                                int dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(pos && neg && out && rows >= 0 && C > 0, "odit_cfg_combine: bad arguments (rows=%lld C=%d)", static_cast<long long>(rows), C);
  ODIT_CHECK_ARG(dtype == ODIT_BF16 || dtype == ODIT_F16, "odit_cfg_combine: dtype must be bf16 or f16, got %d", dtype);
  if (normalize && (C % 8 != 0 || !aligned16(pos) || !aligned16(neg) || !aligned16(out))) {
    set_error("odit_cfg_combine: rows must be 16-byte aligned and a multiple of 8 long (C=%d)", C);
    return ODIT_ENOTSUP;
  }
  if (rows == 0) return ODIT_OK;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  ODIT_DISPATCH_DTYPE(dtype, T, {
    if (sizeof(T) == 2) {
      using H = std::conditional_t<sizeof(T) == 2, T, bf16_t>;
      const H *p = static_cast<const H*>(pos), *q = static_cast<const H*>(neg);
      if (normalize)
        cfg_combine_norm_kernel<H><<<blocks_for(rows * kRowLanes), kBlock, 0, s>>>(p, q, static_cast<H*>(out), rows, C, scale);
      else
        cfg_combine_kernel<H><<<blocks_for(rows * C), kBlock, 0, s>>>(p, q, static_cast<H*>(out), rows * C, scale);
    }
  });
  return check_launch("odit_cfg_combine");
}

extern "C" int odit_euler_step(const void* x, const void* v, void* out, int64_t n, float dt, int dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(x && v && out && n >= 0, "odit_euler_step: bad arguments (n=%lld)", static_cast<long long>(n));
  if (n == 0) return ODIT_OK;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  ODIT_DISPATCH_DTYPE(dtype, T, {
    euler_step_kernel<T><<<blocks_for(n), kBlock, 0, s>>>(static_cast<const T*>(x), static_cast<const T*>(v), static_cast<T*>(out), n, dt);
  });
  return check_launch("odit_euler_step");
}
