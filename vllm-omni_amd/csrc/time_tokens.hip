// Timestep embedding and modulation parameters of a timestep per token: temb = linear_2(silu(linear_1(sinusoid of t))), proj =
// time_proj(silu(temb)) for n tokens. Where an image or a first frame is given, its tokens have one timestep and the others
// another, and n rows of these projections are two rows over and over (width 5120, 2706 tokens: 1 TFLOP, 770 us, an eighth of a
// step of three blocks). So the distinct timesteps are found on the device (up to kRows, no synchronisation), those rows go
// through the kernels for few rows, which stream the weights once (80 us), and every token is told which are its own. Launches of the tile kernel for
// all tokens stand in between and end at once where that went well; where it did not, the launches for few rows make those launches' operands instead
// (the sinusoids, the SiLU), so that the calls that gain nothing pay for the search and for nothing else: seven launches, six without any of this. us,
// every token's rows formed / two timesteps / all different: n=1000, width 5120 319 / 89 / 325; 2706, 5120 773 / 89 / 779; 9000, 3072 935 / 51 / 943;
// 32760, 5120 8650 / 234 / 8615; where the products are small the search and a tile kernel that is not always the best one for them show: 500, 3072 95 /
// - / 108, 2161, 1536 104 / - / 124, 16 us at most. (With launches of their own for the operands and a search of 26 us, 319 / 99 / 343, 773 / 100 / 790, 931 / 63 / 955.)
#include "gemm_bf16.h"
#include "time_sinusoid.h"
#include "time_tokens.h"

namespace odit {
namespace {

constexpr int kRows = 4;  // what linear_stream_kernel takes at a time
constexpr int kThreads = 1024, kEach = 8;

// What the device knows of the timesteps: `few` distinct ones, or 0 of them where there are more than kRows. `value`: they, padded with the first.
struct TimeGroups {
  int few;
  int pad[3];
  float value[kRows];  // (of the timesteps' type, from the first byte)
};
constexpr size_t kHeadBytes = 256;  // (every part on whole cache lines: rows 64 bytes off made the products 16 % slower)
static_assert(sizeof(TimeGroups) <= kHeadBytes, "");

// One workgroup: timesteps that are none of those found so far, until there is none or they are too many. `index`: each token's number among them, its
// own where they are too many. A round is the compares, one candidate of each wavefront by ballot, one barrier, and every wavefront going through the
// candidates: the launch is this chain, of one round where all are different. us, 2706 tokens, two timesteps / all different: 6.0 / 5.1; one timestep a
// round 5.6 / 10.1; one a round by an LDS minimum over all lanes (64 lanes at one address, 4.5 a round) and two barriers 11.2 / 25.7.
template <typename TT, typename Bits>
__global__ __launch_bounds__(kThreads) void time_groups_kernel(const Bits* __restrict__ t, int n, TimeGroups* __restrict__ g, int* __restrict__ index) {
  constexpr int kWaves = kThreads / 64;
  __shared__ int has[2][kWaves];  // (by turns: a wavefront may be a round ahead of one that still reads)
  __shared__ Bits found[2][kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // (the first trip's timesteps stay in registers)
  Bits v[kRows], held[kEach];
#pragma unroll
  for (int e = 0; e < kEach; ++e) held[e] = t[min(tid + e * kThreads, n - 1)];
  int count = 0, from = tid;  // what a thread has before `from` is known, and stays so
  for (int k = 0; count <= kRows; ++k) {  // (a round finds one timestep at least, or ends)
    bool mine = false;
    Bits its = 0;
    while (from < n) {
      Bits b[kEach];
#pragma unroll
      for (int e = 0; e < kEach; ++e) b[e] = from == tid ? held[e] : t[min(from + e * kThreads, n - 1)];
#pragma unroll
      for (int e = kEach - 1; e >= 0; --e) {
        bool known = false;
#pragma unroll
        for (int j = 0; j < kRows; ++j) known |= j < count && b[e] == v[j];
        if (!known) {
          mine = true;
          its = b[e];
        }
      }
      if (mine) break;
      from += kThreads * kEach;
    }
    const uint64_t who = __ballot(mine);
    if (lane == 0) has[k & 1][wave] = who != 0;
    if (mine && (who & ((1ull << lane) - 1)) == 0) found[k & 1][wave] = its;
    __syncthreads();
    uint64_t waves = __ballot(lane < kWaves && has[k & 1][lane % kWaves] != 0);
    if (waves == 0) break;  // (the same for all)
    const Bits theirs = found[k & 1][lane % kWaves];
    while (waves != 0 && count <= kRows) {  // (every pass takes one timestep out, its own at least)
      const int w = __builtin_ctzll(waves);
      const Bits next = static_cast<Bits>(__builtin_amdgcn_readlane(static_cast<int>(theirs), w));
#pragma unroll
      for (int j = 0; j < kRows; ++j)
        if (j == count) v[j] = next;
      ++count;
      waves &= ~(__ballot(theirs == next));
    }
  }
  const int few = count <= kRows ? count : 0;
  if (tid == 0) {
    g->few = few;
    Bits* const out = reinterpret_cast<Bits*>(g->value);
#pragma unroll
    for (int j = 0; j < kRows; ++j) out[j] = j < count ? v[j] : v[0];
  }
  for (int i0 = tid; i0 < n; i0 += kThreads * kEach) {
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int i = i0 + e * kThreads;
      if (i >= n) break;
      const Bits b = i0 == tid ? held[e] : t[i];
      int at = 0;
#pragma unroll
      for (int j = 1; j < kRows; ++j) at = j < few && b == v[j] ? j : at;
      index[i] = few == 0 ? i : at;
    }
  }
}

template <typename T, typename TT>
__global__ __launch_bounds__(256) void token_sinusoid_kernel(const TT* __restrict__ t, T* __restrict__ out, int64_t n, int half, float neg_log_period, float scale) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n * half; i += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t row = i / half;
    const int j = static_cast<int>(i - row * half);
    time_sinusoid<T>(t[row], j, half, neg_log_period, scale, 1.f, out[row * 2 * half + j], out[row * 2 * half + half + j]);
  }
}

struct TokenScratch {
  size_t few, all[3], bytes;
};
TokenScratch token_scratch(int64_t n, int K, int C) {
  TokenScratch s;
  size_t at = kHeadBytes;
  auto take = [&](size_t bytes) {
    const size_t was = at;
    at += (bytes + 255) / 256 * 256;
    return was;
  };
  s.few = take(static_cast<size_t>(kRows) * C * 2);
  s.all[0] = take(static_cast<size_t>(n) * K * 2);
  s.all[1] = take(static_cast<size_t>(n) * C * 2);
  s.all[2] = take(static_cast<size_t>(n) * C * 2);
  s.bytes = at;
  return s;
}
unsigned blocks(int64_t items) { return static_cast<unsigned>(items < 4096 * 256 ? (items + 255) / 256 : 4096); }

template <typename T, typename TT>
int run(const odit_time_tokens_args& a, const TokenScratch& at, char* s, void* workspace, size_t workspace_bytes, int t_dtype, int dtype, hipStream_t stream) {
  const int n = a.n;
  TimeGroups* const g = reinterpret_cast<TimeGroups*>(s);
  const int* const few = &g->few;
  void *const h4 = s + at.few, *const rows = s + at.all[0], *const hidden = s + at.all[1], *const act = s + at.all[2];
  using Bits = std::conditional_t<sizeof(TT) == 4, uint32_t, uint16_t>;
  // nothing is launched unless all of it can be
  auto tile = [&](const void* x, int i, void* out, int N, int K, bool ask) {
    return linear_tile_unless(x, a.w[i], a.bias[i], out, n, N, K, a.ldw[i], dtype, workspace, workspace_bytes, few, ask, stream);
  };
  const int64_t vecs = static_cast<int64_t>(n) * (a.C / 8);
  auto some = [&](const void* x, int i, void* out, int N, const void* of_all, bool ask) {
    return linear_few_or(x, a.w[i], a.bias[i], out, kRows, N, a.C, a.ldw[i], dtype, FewOr{few, of_all, act, vecs}, ask, stream);
  };
  // (the first product, K of 256, is a fiftieth of the work: by any kernel, then for all tokens in either case)
  const bool first_tile = tile(rows, 0, hidden, a.C, a.K, true) == ODIT_OK;
  for (const bool ask : {true, false}) {
    int rc = ODIT_OK;
    auto go = [&](auto&& f) { if (rc == ODIT_OK) rc = f(); };
    if (!ask) {
      time_groups_kernel<TT, Bits><<<1, kThreads, 0, stream>>>(static_cast<const Bits*>(a.t), n, g, a.index);
      rc = check_launch("odit_time_tokens (distinct timesteps)");
    }
    go([&] { return time_linear_or(g->value, a.w[0], a.bias[0], h4, kRows, a.C, a.K, a.ldw[0], a.neg_log_period, a.scale, t_dtype, dtype,
                                   FewOr{few, a.t, first_tile ? rows : nullptr, n}, ask, stream); });
    if (first_tile) {
      go([&] { return tile(rows, 0, hidden, a.C, a.K, ask); });
    } else if (!ask) {
      go([&] {
        token_sinusoid_kernel<T, TT><<<blocks(static_cast<int64_t>(n) * (a.K / 2)), 256, 0, stream>>>(static_cast<const TT*>(a.t), static_cast<T*>(rows), n,
                                                                                                      a.K / 2, a.neg_log_period, a.scale);
        return check_launch("odit_time_tokens (rows)");
      });
      go([&] { return odit_linear_rows(rows, a.w[0], a.bias[0], hidden, nullptr, nullptr, n, a.C, a.K, a.K, a.ldw[0], a.C, 0,
                                       a.bias[0] != nullptr ? ODIT_EPI_BIAS : ODIT_EPI_NONE, dtype, dtype, 0, 0, 0, workspace, workspace_bytes, stream); });
    }
    go([&] { return some(h4, 1, a.temb, a.C, hidden, ask); });
    go([&] { return tile(act, 1, a.temb, a.C, a.C, ask); });
    go([&] { return some(a.temb, 2, a.proj, a.P, a.temb, ask); });
    go([&] { return tile(act, 2, a.proj, a.P, a.C, ask); });
    if (rc != ODIT_OK) return rc;
  }
  return ODIT_OK;
}

}  // namespace
}  // namespace odit

extern "C" size_t odit_time_tokens_bytes(int n, int K, int C) {
  return n > 0 && K > 0 && C > 0 ? odit::token_scratch(n, K, C).bytes : 0;
}

extern "C" int odit_time_tokens(const odit_time_tokens_args* args, void* scratch, size_t scratch_bytes, int t_dtype, int dtype, void* workspace,
                                size_t workspace_bytes, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(args != nullptr, "odit_time_tokens: null arguments");
  const odit_time_tokens_args& a = *args;
  ODIT_CHECK_ARG(a.t && a.temb && a.proj && a.index && a.n >= kRows && a.n < (1 << 30) && a.K > 0 && a.K % 2 == 0 && a.C > 0 && a.P > 0, "odit_time_tokens: bad arguments (n=%d K=%d C=%d P=%d)", a.n,
                 a.K, a.C, a.P);
  for (int i = 0; i < 3; ++i) ODIT_CHECK_ARG(a.w[i] != nullptr && a.ldw[i] >= (i == 0 ? a.K : a.C), "odit_time_tokens: weight %d", i);
  ODIT_CHECK_ARG(t_dtype >= ODIT_BF16 && t_dtype <= ODIT_F32, "odit_time_tokens: dtype code %d", t_dtype);
  if ((dtype != ODIT_BF16 && dtype != ODIT_F16) || a.C % 8 != 0 || a.P % 8 != 0 || !aligned16(a.temb) || !aligned16(a.proj)) {
    set_error("odit_time_tokens: takes 16-bit types and 16-byte aligned rows (C=%d P=%d)", a.C, a.P);
    return ODIT_ENOTSUP;
  }
  const TokenScratch at = token_scratch(a.n, a.K, a.C);
  if (scratch == nullptr || scratch_bytes < at.bytes || (reinterpret_cast<uintptr_t>(scratch) & 255) != 0) {
    set_error("odit_time_tokens: %zu bytes of 256-byte aligned scratch needed, %zu given", at.bytes, scratch_bytes);
    return ODIT_EWORKSPACE;
  }
  const hipStream_t s = static_cast<hipStream_t>(stream);
  char* const p = static_cast<char*>(scratch);
#define ODIT_TOKENS(T, TT) return run<T, TT>(a, at, p, workspace, workspace_bytes, t_dtype, dtype, s)
  if (dtype == ODIT_BF16) {
    if (t_dtype == ODIT_BF16) ODIT_TOKENS(bf16_t, bf16_t);
    if (t_dtype == ODIT_F16) ODIT_TOKENS(bf16_t, f16_t);
    ODIT_TOKENS(bf16_t, float);
  }
  if (t_dtype == ODIT_BF16) ODIT_TOKENS(f16_t, bf16_t);
  if (t_dtype == ODIT_F16) ODIT_TOKENS(f16_t, f16_t);
  ODIT_TOKENS(f16_t, float);
#undef ODIT_TOKENS
}
