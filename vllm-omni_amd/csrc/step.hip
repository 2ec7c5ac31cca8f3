// The small work around the transformer in a denoise step: the timestep sinusoid, the rotary tables of the position ids, the gate
// rows of the blocks, the stacked branches of CFG, their combination and the Euler update.
// Every tensor here is a few KB to a few MB, so what bounds it is the number of launches and the host time of each: as torch
// operations the first and the last two were 10, 7 and 5 launches (about 2 us each on the GPU and 4 to 8 us on the host); here
// each is one.
// Every intermediate is rounded where the torch expression rounds it, with no contraction of multiply and add.
#include "odit_common.h"
#include "time_sinusoid.h"

#pragma clang fp contract(off)

namespace odit {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxBlocks = 4096;

// out[i, :] = cos | sin (time_sinusoid.h) of every frequency
template <typename TT, typename T>
__global__ __launch_bounds__(kBlock) void time_sinusoid_kernel(const TT* __restrict__ t, T* __restrict__ out, int64_t n, int half,
                                                               float neg_log_period, float scale, float pre) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n * half; i += static_cast<int64_t>(gridDim.x) * kBlock) {
    const int64_t row = i / half;
    const int j = static_cast<int>(i - row * half);
    time_sinusoid<T>(t[row], j, half, neg_log_period, scale, pre, out[row * 2 * half + j], out[row * 2 * half + half + j]);
  }
}

// Rows copied and padded, up to 16 tensors in a launch. As torch operations the branches of a CFG pair were three concatenations, with prompts of
// unequal length ten launches, one after the other in front of a step's first projection: 19 and 58 us a step, the host's, here 10 and 11
// (1024 latent tokens and 171 + 171, 171 + 23 text tokens of width 3584). A workgroup has kPadEach granules of one piece for each lane: the widest power of two up to 16 bytes that divides the piece's addresses and lengths.
constexpr int kPadEach = 4;
struct PadPiece {
  const char* src;
  char* dst;
  int64_t src_pitch;
  uint32_t granules, copy, pitch, first;  // granules in all, of a row that are copied, of a row; first workgroup
  uint8_t log2, head, tail;
};
struct PadPieces {
  PadPiece p[ODIT_PAD_PIECES];
  int n;
};
template <typename V> __device__ __forceinline__ V filled(uint32_t byte) { return static_cast<V>(static_cast<uint64_t>(byte) * 0x0101010101010101ull); }
template <> __device__ __forceinline__ u32x4 filled<u32x4>(uint32_t byte) { const uint32_t w = byte * 0x01010101u; return u32x4{w, w, w, w}; }
template <typename V> __device__ __forceinline__ void pad_granules(const PadPiece& p, uint32_t g0) {
  V v[kPadEach];
#pragma unroll
  for (int i = 0; i < kPadEach; ++i) {
    const uint32_t g = g0 + i * kBlock, row = g / p.pitch, at = g - row * p.pitch;
    if (g >= p.granules || at >= p.copy) v[i] = filled<V>(p.tail);
    else if (p.src == nullptr) v[i] = filled<V>(p.head);
    else v[i] = *reinterpret_cast<const V*>(p.src + row * p.src_pitch + static_cast<int64_t>(at) * sizeof(V));
  }
#pragma unroll
  for (int i = 0; i < kPadEach; ++i)
    if (g0 + i * kBlock < p.granules) reinterpret_cast<V*>(p.dst)[g0 + i * kBlock] = v[i];
}
__global__ __launch_bounds__(kBlock) void pad_rows_kernel(const PadPieces a) {
  int i = 0;
  while (i + 1 < a.n && blockIdx.x >= a.p[i + 1].first) ++i;  // (launch-uniform per workgroup)
  const PadPiece& p = a.p[i];
  const uint32_t g0 = (blockIdx.x - p.first) * (kBlock * kPadEach) + threadIdx.x;
  switch (p.log2) {
    case 4: pad_granules<u32x4>(p, g0); break;
    case 3: pad_granules<uint64_t>(p, g0); break;
    case 2: pad_granules<uint32_t>(p, g0); break;
    case 1: pad_granules<uint16_t>(p, g0); break;
    default: pad_granules<uint8_t>(p, g0); break;
  }
}

// Rotary tables of position ids, text rows before image rows: out[row, j] = cos | sin of id[row, axis] * theta^(-2 k / d), k the
// column j within its axis, everything in float64 up to the rounding to float32. As torch operations this was 33 launches
// (4 to 7 us each, 150 us per step, and as much host time again); as one launch it takes about 6 us at 4608 rows of 64 columns,
// bound by the float64 pow, sin and cos. A thread keeps one column, so the pow is paid once for kRopeRows / 4 rows.
constexpr int kMaxAxes = 4, kRopeRows = 16;
struct RopeAxes {
  int count, half;           // axes, columns in all
  int start[kMaxAxes + 1];   // first column of every axis
};
template <typename T>
__global__ __launch_bounds__(kBlock) void rope_tables_kernel(const T* __restrict__ txt, int64_t n_txt, const T* __restrict__ img,
                                                             int64_t n, float* __restrict__ cos_out, float* __restrict__ sin_out,
                                                             RopeAxes ax, double theta) {
  const int64_t row_end = min(n, (static_cast<int64_t>(blockIdx.x) + 1) * kRopeRows);
  for (int j = threadIdx.x % 64; j < ax.half; j += 64) {
    int a = 0;
    while (a + 1 < ax.count && j >= ax.start[a + 1]) ++a;
    const int d = 2 * (ax.start[a + 1] - ax.start[a]);
    const double inv = 1.0 / pow(theta, static_cast<double>(2 * (j - ax.start[a])) / static_cast<double>(d));
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * kRopeRows + threadIdx.x / 64; row < row_end; row += kBlock / 64) {
      const T* id = row < n_txt ? txt + row * ax.count : img + (row - n_txt) * ax.count;
      const double ang = static_cast<double>(to_float(id[a])) * inv;
      double c, s;
      sincos(ang, &s, &c);
      cos_out[row * ax.half + j] = static_cast<float>(c);
      sin_out[row * ax.half + j] = static_cast<float>(s);
    }
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

// gates[b, i, c] = mods[b, 3 i C + 2 C + c] and gated = gates * bias_i[c] in float32, for the n gated projections of a model's
// blocks: the last third of each modulation triple and the projection's own bias, wherever that lies. As torch operations (two
// conversions, the stacking of the biases and the product) this was four launches per step, 9 us on the GPU at 8
// projections of 256 and some 30 on the host (a four-step run of the smallest model: 825 us, 735 with the one launch); the one launch
// takes 2.6 us there and 5.0 with 48 projections of 3072. EPV elements a lane.
constexpr int kGateRows = 256;  // pointers that one launch carries (2 of 4 KB of arguments)
struct GateBiases { const void* p[kGateRows]; };
template <typename T, int EPV>
__global__ __launch_bounds__(kBlock) void gate_rows_kernel(const GateBiases bias, const T* __restrict__ mods, int64_t mods_b, float* __restrict__ gates,
                                                           float* __restrict__ gated, int first, int n, int C) {
  const int i = blockIdx.y, b = blockIdx.z, c = (blockIdx.x * kBlock + threadIdx.x) * EPV;
  if (c >= C) return;
  const T* m = mods + b * mods_b + (static_cast<int64_t>(first + i) * 3 + 2) * C + c;
  const T* w = static_cast<const T*>(bias.p[i]) + c;
  const int64_t at = (static_cast<int64_t>(b) * n + first + i) * C + c;
  struct alignas(EPV * sizeof(T)) Vec { T e[EPV]; };
  const Vec mv = *reinterpret_cast<const Vec*>(m), wv = *reinterpret_cast<const Vec*>(w);
  struct alignas(EPV * 4) Out { float e[EPV]; } g, gb;
#pragma unroll
  for (int j = 0; j < EPV; ++j) {
    g.e[j] = to_float(mv.e[j]);
    gb.e[j] = g.e[j] * to_float(wv.e[j]);
  }
  *reinterpret_cast<Out*>(gates + at) = g;
  *reinterpret_cast<Out*>(gated + at) = gb;
}

int blocks_for(int64_t threads) {
  const int64_t b = (threads + kBlock - 1) / kBlock;
  return static_cast<int>(b < kMaxBlocks ? b : kMaxBlocks);
}

template <typename TT, typename T>
int launch_sinusoid(const void* t, void* out, int64_t n, int half, float neg_log_period, float scale, float pre, hipStream_t s) {
  time_sinusoid_kernel<TT, T><<<blocks_for(n * half), kBlock, 0, s>>>(static_cast<const TT*>(t), static_cast<T*>(out), n, half,
                                                                     neg_log_period, scale, pre);
  return check_launch("odit_time_sinusoid");
}

}  // namespace
}  // namespace odit

extern "C" int odit_time_sinusoid(const void* t, void* out, int64_t n, int dim, float neg_log_period, float scale, float pre,
                                  int t_dtype, int out_dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(t && out && n >= 0 && dim > 0 && dim % 2 == 0, "odit_time_sinusoid: needs t, out and an even dim (n=%lld dim=%d)",
                 static_cast<long long>(n), dim);
  if (n == 0) return ODIT_OK;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  ODIT_DISPATCH_DTYPE(t_dtype, TT, {
    ODIT_DISPATCH_DTYPE(out_dtype, T, { return launch_sinusoid<TT, T>(t, out, n, dim / 2, neg_log_period, scale, pre, s); });
  });
  return ODIT_OK;
}

extern "C" int odit_rope_tables(const void* txt_ids, int64_t n_txt, const void* img_ids, int64_t n_img, float* cos_out,
                                float* sin_out, const int* axes_dim, int n_axes, double theta, int dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(n_txt >= 0 && n_img >= 0 && (txt_ids || n_txt == 0) && (img_ids || n_img == 0) && cos_out && sin_out && axes_dim &&
                     n_axes >= 1 && n_axes <= kMaxAxes && theta > 0,
                 "odit_rope_tables: bad arguments (rows %lld + %lld, %d axes)", static_cast<long long>(n_txt),
                 static_cast<long long>(n_img), n_axes);
  RopeAxes ax{};
  ax.count = n_axes;
  for (int i = 0; i < n_axes; ++i) {
    ODIT_CHECK_ARG(axes_dim[i] > 0 && axes_dim[i] % 2 == 0, "odit_rope_tables: axis widths must be even, got %d", axes_dim[i]);
    ax.start[i + 1] = ax.start[i] + axes_dim[i] / 2;
  }
  ax.half = ax.start[n_axes];
  const int64_t n = n_txt + n_img;
  if (n == 0) return ODIT_OK;
  const int64_t blocks = (n + kRopeRows - 1) / kRopeRows;
  ODIT_CHECK_ARG(blocks <= (1 << 24), "odit_rope_tables: too many rows (%lld)", static_cast<long long>(n));
  ODIT_DISPATCH_DTYPE(dtype, T, {
    rope_tables_kernel<T><<<static_cast<int>(blocks), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const T*>(txt_ids), n_txt, static_cast<const T*>(img_ids), n, cos_out, sin_out, ax, theta);
  });
  return check_launch("odit_rope_tables");
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

extern "C" int odit_pad_rows(const odit_pad_piece* pieces, int n, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(n >= 0 && n <= ODIT_PAD_PIECES && (pieces != nullptr || n == 0), "odit_pad_rows: %d pieces, at most %d", n, ODIT_PAD_PIECES);
  PadPieces a;
  a.n = 0;
  uint64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    const odit_pad_piece& s = pieces[i];
    ODIT_CHECK_ARG(s.dst != nullptr && s.rows >= 0 && s.copy >= 0 && s.pitch >= s.copy && s.src_pitch >= 0, "odit_pad_rows: piece %d is bad", i);
    if (s.rows == 0 || s.pitch == 0) continue;
    uint64_t all = reinterpret_cast<uintptr_t>(s.dst) | static_cast<uint64_t>(s.copy) | static_cast<uint64_t>(s.pitch) | 16u;
    if (s.src != nullptr) all |= reinterpret_cast<uintptr_t>(s.src) | static_cast<uint64_t>(s.rows > 1 ? s.src_pitch : 0);
    const int log2 = __builtin_ctzll(all);
    const int64_t pitch = s.pitch >> log2;
    if (pitch >= (1ll << 31) || s.rows >= (1ll << 31) || s.rows * pitch >= (1ll << 31)) {
      set_error("odit_pad_rows: piece %d has more than 2^31 granules", i);
      return ODIT_ENOTSUP;
    }
    PadPiece& p = a.p[a.n++];
    p = PadPiece{static_cast<const char*>(s.src), static_cast<char*>(s.dst), s.src_pitch, static_cast<uint32_t>(s.rows * pitch),
                 static_cast<uint32_t>(s.copy >> log2), static_cast<uint32_t>(pitch), static_cast<uint32_t>(blocks), static_cast<uint8_t>(log2), s.head,
                 s.tail};
    blocks += (p.granules + kBlock * kPadEach - 1) / (kBlock * kPadEach);
  }
  if (a.n == 0) return ODIT_OK;
  pad_rows_kernel<<<static_cast<unsigned>(blocks), kBlock, 0, static_cast<hipStream_t>(stream)>>>(a);
  return check_launch("odit_pad_rows");
}

extern "C" int odit_gate_rows(const void* const* bias, int n, const void* mods, int64_t mods_batch_stride, int B, int C, float* gates,
                              float* gated, int dtype, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(bias && mods && gates && gated && n >= 0 && B >= 0 && B < 65536 && C > 0 && C < (1 << 30) && mods_batch_stride >= 0,
                 "odit_gate_rows: bad arguments (n=%d B=%d C=%d)", n, B, C);
  ODIT_CHECK_ARG(dtype == ODIT_BF16 || dtype == ODIT_F16, "odit_gate_rows: dtype code %d", dtype);
  if (n == 0 || B == 0) return ODIT_OK;
  bool wide = C % 4 == 0 && mods_batch_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(mods) & 7) == 0 && aligned16(gates) && aligned16(gated);
  for (int i = 0; i < n; ++i) {
    ODIT_CHECK_ARG(bias[i] != nullptr, "odit_gate_rows: bias %d is null", i);
    wide = wide && (reinterpret_cast<uintptr_t>(bias[i]) & 7) == 0;
  }
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int per_block = kBlock * (wide ? 4 : 1);
  for (int first = 0; first < n; first += kGateRows) {
    const int rows = n - first < kGateRows ? n - first : kGateRows;
    GateBiases p{};
    for (int i = 0; i < rows; ++i) p.p[i] = bias[first + i];
    const dim3 grid((C + per_block - 1) / per_block, rows, B);
#define ODIT_GATE_ROWS(T)                                                                                                         \
  do {                                                                                                                            \
    if (wide) gate_rows_kernel<T, 4><<<grid, kBlock, 0, s>>>(p, static_cast<const T*>(mods), mods_batch_stride, gates, gated, first, n, C); \
    else gate_rows_kernel<T, 1><<<grid, kBlock, 0, s>>>(p, static_cast<const T*>(mods), mods_batch_stride, gates, gated, first, n, C);      \
  } while (0)
    if (dtype == ODIT_BF16) ODIT_GATE_ROWS(bf16_t);
    else ODIT_GATE_ROWS(f16_t);
#undef ODIT_GATE_ROWS
    const int rc = check_launch("odit_gate_rows");
    if (rc != ODIT_OK) return rc;
  }
  return ODIT_OK;
}
