// Dense projections with fused epilogues: y = x W^T (+ bias) with, in the GEMM's own epilogue,
//   * GELU(tanh)                              (MLP up-projection: no separate activation pass)
//   * out = residual + gate * (x W^T + bias)  (attention / MLP output projections: no separate
//                                              gated-residual pass)
// Which kernel runs is decided here per call. Few rows: the hand-written stream-K kernel (gemm_bf16.hip) where the reduction is
// long, and a kernel for products that are small altogether (gemm_small.hip). Many rows: the hand-written tile kernel
// (gemm_tile.h) or hipBLASLt's MFMA kernels, by expected time. The two streams of a dual-stream block: one launch of a
// hand-written kernel, or two calls, by expected time (odit_linear_pair), with what follows a projection to heads at its end where
// that is expected to be faster (odit_linear_heads). For the library this file sets the problem up so that
// its epilogue does the elementwise work (bias vector, activation, a per-output-feature alpha vector for the gate, beta = 1 on the
// residual), keeps problem descriptors per thread, chooses among the library's candidates for long reductions by expected time, and
// has an explicit tuning call that times the library's kernels and the hand-written ones for one problem and remembers the fastest.
//
// Row-major y[M,N] = x[M,K] W[N,K]^T is the column-major product D(N x M) = op(A) B with A = W stored
// K x N (ld = ldw, transposed), B = x stored K x M (ld = ldx): the bias and the alpha vector run along
// D's rows, i.e. along the N output features, as needed.
#include "odit_common.h"
#include "gemm_epilogue.h"
#include "time_tokens.h"

#include <hipblaslt/hipblaslt.h>
#include <hipblaslt/hipblaslt-ext.hpp>

#include <algorithm>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

namespace odit {

// alpha[n] = gate[n], gbias[n] = gate[n] * bias[n], both fp32, for the gated-residual epilogue
template <typename T, typename TG>
__global__ __launch_bounds__(256) void gate_prep_kernel(const TG* __restrict__ gate, const T* __restrict__ bias,
                                                         float* __restrict__ alpha, float* __restrict__ gbias, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const float g = gate ? to_float(gate[i]) : 1.f;
    alpha[i] = g;
    gbias[i] = bias ? g * to_float(bias[i]) : 0.f;
  }
}

struct LinKey {
  int dev, m, n, k, epi, dtype;
  int64_t lda, ldb, ldc, ldd;
  bool operator==(const LinKey& o) const {
    return dev == o.dev && m == o.m && n == o.n && k == o.k && epi == o.epi && dtype == o.dtype &&
           lda == o.lda && ldb == o.ldb && ldc == o.ldc && ldd == o.ldd;
  }
};
struct LinKeyHash {
  size_t operator()(const LinKey& k) const {
    size_t h = 1469598103934665603ull;
    auto mix = [&](uint64_t v) { h = (h ^ v) * 1099511628211ull; };
    mix(k.dev); mix(k.m); mix(k.n); mix(k.k); mix(k.epi); mix(k.dtype);
    mix(static_cast<uint64_t>(k.lda)); mix(static_cast<uint64_t>(k.ldb));
    mix(static_cast<uint64_t>(k.ldc)); mix(static_cast<uint64_t>(k.ldd));
    return h;
  }
};

struct LinPlan {
  hipblasLtMatmulDesc_t desc = nullptr;
  hipblasLtMatrixLayout_t a = nullptr, b = nullptr, c = nullptr, d = nullptr;
  hipblasLtMatmulAlgo_t algo;
  size_t algo_ws = 0;
  bool have_algo = false;
  bool tuned = false;
  int passed = 0;  // the library's first choice is never run (lin_sound): it would have summed every tile whole (1), or split some among passed - 1 workers
  float us = 0;  // expected time of a kernel that was ranked, 0: not known
};

// One hipBLASLt handle and one plan cache per host thread: plans are mutated per call (bias and
// alpha-vector pointers), so they are never shared between threads.
struct LinState {
  hipblasLtHandle_t handle[64] = {nullptr};
  std::unordered_map<LinKey, LinPlan, LinKeyHash> plans;
};
static thread_local LinState g_lin;

// What a tuning call found for a problem: the fastest kernel (0 the library's, which is in the plan of the thread that tuned; else
// a hand-written one, see lin_candidate) and its time. Key: the whole problem, rows_per_gate in the lda field, and whether there
// was scratch. Process-wide and kept for the life of the process: every host thread sees what any thread has measured, and the
// record outlives the per-thread descriptor cache.
struct Tuned { int kind; float us; };
static std::mutex g_engine_mu;
static std::unordered_map<LinKey, Tuned, LinKeyHash> g_tuned;

// Library kernels chosen ahead of time for plain projections (odit_linear_prefer): (N, M, K, element type) -> the
// library's own solution index. Few entries, read when a problem is first seen.
struct Preferred { int m, n, k, dtype, solution; };
static std::vector<Preferred> g_preferred;  // guarded by g_engine_mu

#define ODIT_LT(call)                                                                      \
  do {                                                                                     \
    const hipblasStatus_t st__ = (call);                                                   \
    if (st__ != HIPBLAS_STATUS_SUCCESS) {                                                  \
      set_error("odit_linear: %s failed with hipBLAS status %d", #call, static_cast<int>(st__)); \
      return ODIT_ELAUNCH;                                                                 \
    }                                                                                      \
  } while (0)

static int lin_handle(int dev, hipblasLtHandle_t* out) {
  if (dev < 0 || dev >= 64) { set_error("odit_linear: device index %d out of range", dev); return ODIT_EINVAL; }
  if (g_lin.handle[dev] == nullptr) ODIT_LT(hipblasLtCreate(&g_lin.handle[dev]));
  *out = g_lin.handle[dev];
  return ODIT_OK;
}

static hipDataType lin_type(int dtype) {
  return dtype == ODIT_BF16 ? HIP_R_16BF : (dtype == ODIT_F16 ? HIP_R_16F : HIP_R_32F);
}

static void lin_plan_release(LinPlan& p) {
  if (p.a) hipblasLtMatrixLayoutDestroy(p.a);
  if (p.b) hipblasLtMatrixLayoutDestroy(p.b);
  if (p.c) hipblasLtMatrixLayoutDestroy(p.c);
  if (p.d) hipblasLtMatrixLayoutDestroy(p.d);
  if (p.desc) hipblasLtMatmulDescDestroy(p.desc);
  p = LinPlan{};
}

static int lin_plan_build(const LinKey& key, LinPlan& p) {
  const hipDataType t = lin_type(key.dtype);
  ODIT_LT(hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F));
  const int32_t ta = HIPBLAS_OP_T, tb = HIPBLAS_OP_N;
  ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &ta, sizeof(ta)));
  ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &tb, sizeof(tb)));
  // key.epi = epilogue * 4 + (bias vector in the epilogue ? 1 : 0) + (alpha vector ? 2 : 0); a first-ranked kernel has a plan of its own (+ 0x100)
  const int kind = (key.epi & 0xff) >> 2;
  const bool has_bias = key.epi & 1, alpha_vec = key.epi & 2;
  const bool gelu = kind == ODIT_EPI_GELU_TANH || kind == ODIT_EPI_BIAS_GELU_TANH;
  const uint32_t epi = gelu ? (has_bias ? HIPBLASLT_EPILOGUE_GELU_BIAS : HIPBLASLT_EPILOGUE_GELU)
                            : (has_bias ? HIPBLASLT_EPILOGUE_BIAS : HIPBLASLT_EPILOGUE_DEFAULT);
  ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_EPILOGUE, &epi, sizeof(epi)));
  if (alpha_vec) {
    const int32_t pm = HIPBLASLT_POINTER_MODE_ALPHA_DEVICE_VECTOR_BETA_HOST;
    ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_POINTER_MODE, &pm, sizeof(pm)));
  }
  if (has_bias) {  // the gate-scaled bias that goes with an alpha vector is fp32
    const int32_t bt = alpha_vec ? HIP_R_32F : t;
    ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_DATA_TYPE, &bt, sizeof(bt)));
  }
  // column-major views: A = W (K x N, ld lda), B = x (K x M, ld ldb), C/D = N x M
  ODIT_LT(hipblasLtMatrixLayoutCreate(&p.a, t, key.k, key.n, key.lda));
  ODIT_LT(hipblasLtMatrixLayoutCreate(&p.b, t, key.k, key.m, key.ldb));
  ODIT_LT(hipblasLtMatrixLayoutCreate(&p.c, t, key.n, key.m, key.ldc));
  ODIT_LT(hipblasLtMatrixLayoutCreate(&p.d, t, key.n, key.m, key.ldd));
  return ODIT_OK;
}

static int lin_plan(const LinKey& key, LinPlan** out) {
  auto it = g_lin.plans.find(key);
  if (it != g_lin.plans.end()) { *out = &it->second; return ODIT_OK; }
  // A process sees a few dozen distinct problems; a caller that keeps inventing new ones (changing row
  // counts) must not grow the cache without bound: past the cap everything is rebuilt on demand.
  constexpr size_t kMaxPlans = 512;
  if (g_lin.plans.size() >= kMaxPlans) {
    for (auto& kv : g_lin.plans) lin_plan_release(kv.second);
    g_lin.plans.clear();
  }
  LinPlan p;
  const int rc = lin_plan_build(key, p);
  if (rc != ODIT_OK) {  // nothing half-built stays behind
    lin_plan_release(p);
    return rc;
  }
  auto ins = g_lin.plans.emplace(key, p);
  *out = &ins.first->second;
  return ODIT_OK;
}

// engine bits of the `flags` argument: neither = the hand-written kernel where it takes the problem and is
// expected (or was measured) to win, else the library
static int lin_engine_of(unsigned flags) {
  return (flags & ODIT_LINEAR_LIBRARY) ? 1 : ((flags & ODIT_LINEAR_HANDWRITTEN) ? 2 : 0);
}

struct LinCall {
  const void *x, *w, *bias, *residual, *gate;
  void* out;
  int M, N, K;
  int64_t ldx, ldw, ldo, ldr;
  int epilogue, gate_dtype, dtype;
  void* ws;
  size_t ws_bytes;
  hipStream_t stream;
  bool first = false;    // the library's first-ranked kernel, unless one was tuned (ODIT_LINEAR_FIRST)
  bool no_tile = false;  // untuned, neither the tile nor the small kernel (ODIT_LINEAR_NO_TILE)
  bool clip = false;     // results of f16 clipped (ODIT_LINEAR_CLIP)
};

static bool lin_is_residual(const LinCall& c) {
  return c.epilogue == ODIT_EPI_GATED_RESIDUAL || c.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
}
// the gate has to be turned into fp32 alpha / gate*bias vectors by a helper launch
static bool lin_needs_prep(const LinCall& c) { return c.epilogue == ODIT_EPI_GATED_RESIDUAL && c.gate != nullptr; }

// workspace split: [0, 8N rounded to 256) gate vectors (when a helper launch makes them), the rest for
// the library
static size_t lin_gate_bytes(const LinCall& c) {
  return lin_needs_prep(c) ? ((static_cast<size_t>(c.N) * 8 + 255) / 256) * 256 : 0;
}

static LinKey lin_plan_key(int dev, const LinCall& c) {
  const bool gated = lin_is_residual(c);
  return LinKey{dev, c.M, c.N, c.K, c.epilogue * 4 + (c.bias != nullptr ? 1 : 0) + (gated && c.gate != nullptr ? 2 : 0), c.dtype, c.ldw, c.ldx,
                gated ? c.ldr : c.ldo, c.ldo};
}

// the handle, and the plan of the problem (as many launches as there are groups of rows share it)
static int lin_find_plan(const LinCall& c, hipblasLtHandle_t* h, LinPlan** plan) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { set_error("odit_linear: hipGetDevice failed"); return ODIT_ELAUNCH; }
  const int rc = lin_handle(dev, h);
  if (rc != ODIT_OK) return rc;
  LinKey key = lin_plan_key(dev, c);
  if (c.first) {  // unless a tuning call has found this problem's fastest kernel: what it chose runs
    const auto it = g_lin.plans.find(key);
    if (it == g_lin.plans.end() || !it->second.tuned) key.epi |= 0x100;
  }
  return lin_plan(key, plan);
}

static int lin_prepare(const LinCall& c, hipblasLtHandle_t* h, LinPlan** plan, const void** alpha_ptr,
                       const void** c_ptr, void** lib_ws, size_t* lib_ws_bytes) {
  int rc = lin_find_plan(c, h, plan);
  if (rc != ODIT_OK) return rc;
  const bool gated = lin_is_residual(c);
  const bool prep = lin_needs_prep(c);
  const bool alpha_vec = gated && c.gate != nullptr;
  const bool has_bias = c.bias != nullptr;
  const size_t gb = lin_gate_bytes(c);
  if (gb > c.ws_bytes) {
    set_error("odit_linear: workspace of %zu bytes cannot hold the %zu bytes of gate vectors", c.ws_bytes, gb);
    return ODIT_EWORKSPACE;
  }
  *lib_ws = c.ws ? static_cast<char*>(c.ws) + gb : nullptr;
  *lib_ws_bytes = c.ws ? c.ws_bytes - gb : 0;
  static const float one = 1.f;
  *alpha_ptr = &one;
  *c_ptr = c.out;
  LinPlan& p = **plan;
  if (gated) *c_ptr = c.residual;
  if (prep) {
    float* alpha = static_cast<float*>(c.ws);
    float* gbias = alpha + c.N;
    const dim3 grid((c.N + 255) / 256);
#define ODIT_GATE_PREP(T, TG)                                                                        \
  hipLaunchKernelGGL((gate_prep_kernel<T, TG>), grid, dim3(256), 0, c.stream, static_cast<const TG*>(c.gate), \
                     static_cast<const T*>(c.bias), alpha, gbias, c.N)
    if (c.gate_dtype == ODIT_F32) {
      ODIT_DISPATCH_DTYPE(c.dtype, T, ODIT_GATE_PREP(T, float));
    } else {
      ODIT_DISPATCH_DTYPE(c.dtype, T, ODIT_GATE_PREP(T, T));
    }
#undef ODIT_GATE_PREP
    rc = check_launch("odit_linear (gate vectors)");
    if (rc != ODIT_OK) return rc;
    if (has_bias) {
      const void* bp = gbias;
      ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bp, sizeof(bp)));
    }
    *alpha_ptr = alpha;
  } else {
    if (has_bias) {
      const void* bp = c.bias;
      ODIT_LT(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bp, sizeof(bp)));
    }
    if (alpha_vec) *alpha_ptr = c.gate;  // caller-made fp32 vectors
  }
  return ODIT_OK;
}

// The library's hand-scheduled kernel of 256 x 256 x 64 ("Custom_...", its first choice for most problems of many rows) now and then gives other results for
// the same operands: 8 rows of a tile, those that one of its loads fetches (30 and 31 of each 32 rows of a half), times up to 128 features, off by the size of
// the values themselves. In passes of a block of width 5120 over 65520 rows, five launches of it each, 1 of 100 and 1 of 300; the tile kernel in its place none of
// 600, the library's other kernels in the same passes none. It is left out wherever a kernel is chosen, timed or named.
static bool lin_sound(hipblasLtHandle_t h, hipblasLtMatmulAlgo_t& algo) { return hipblaslt_ext::getKernelNameFromAlgo(h, algo).rfind("Custom", 0) != 0; }

// The solution that odit_linear_prefer named for this problem (a plain projection with bias and dense rows), when the
// library has it and it accepts the problem and the workspace.
static bool lin_preferred_algo(hipblasLtHandle_t h, LinPlan& p, const LinCall& c, size_t lib_ws_bytes) {
  if (c.epilogue != ODIT_EPI_BIAS || c.ldx != c.K || c.ldw != c.K || c.ldo != c.N) return false;
  int solution = -1;
  {
    std::lock_guard<std::mutex> lock(g_engine_mu);
    for (const Preferred& e : g_preferred)
      if (e.m == c.M && e.n == c.N && e.k == c.K && e.dtype == c.dtype) { solution = e.solution; break; }
  }
  if (solution < 0) return false;
  std::vector<int> index{solution};
  std::vector<hipblasLtMatmulHeuristicResult_t> found;
  if (hipblaslt_ext::getAlgosFromIndex(h, index, found) != HIPBLAS_STATUS_SUCCESS || found.empty() || !lin_sound(h, found[0].algo)) return false;
  const float one = 1.f, zero = 0.f;
  size_t need = 0;
  if (hipblaslt_ext::matmulIsAlgoSupported(h, p.desc, &one, p.a, p.b, &zero, p.c, p.d, found[0].algo, need) != HIPBLAS_STATUS_SUCCESS ||
      need > lib_ws_bytes)
    return false;
  p.algo = found[0].algo;
  p.algo_ws = need;
  p.have_algo = true;
  return true;
}

// Macro tile of a library kernel, from its name ("..._MT256x192x64_..."): features x rows x reduction step. Only the
// kernels of the usual wave layout (WG32_8) with steps of 64 count: the others of the same
// tile run 10 to 25 % slower, and the time model below was fitted without them.
static bool lin_macro_tile(const std::string& name, int* features, int* rows, bool* usual) {
  const size_t at = name.find("_MT");
  int step = 0;
  if (at == std::string::npos || sscanf(name.c_str() + at, "_MT%dx%dx%d", features, rows, &step) != 3) return false;
  *usual = step == 64 && name.find("_WG32_8_", at) != std::string::npos;
  return true;
}

// Expected time (us) of a problem on a library kernel of one macro tile: rounds of tiles over the compute units times the
// time of one tile, fitted to 1600 launches (bf16, 1024 <= M <= 13056, the projections of widths 3072 and 5120, last
// round over 0.93 full; residual 9 %). The library divides a last round that is not full between the units (stream-K). At
// K >= 8192 that costs up to a round more than its share of tiles (M=6144, N=3072, K=12288 on 256 x 160 tiles, 1.8
// rounds: 682 us; on 192 x 192, 2.0 rounds: 340), unless the round is at least 0.88 full: then it is left undivided.
static double lin_tile_us(int M, int N, int K, int features, int rows, int cus) {
  const int64_t tiles = static_cast<int64_t>((N + features - 1) / features) * ((M + rows - 1) / rows);
  const int64_t rounds = (tiles + cus - 1) / cus;
  const double share = static_cast<double>(tiles) / cus, last = share - static_cast<double>(rounds - 1);
  const double tile = 2.31 + K * (2.35e-7 * features * rows + 1.26e-5 * (features + rows) + 1.82e-3);
  if (last >= 0.88 || K < 8192) return static_cast<double>(rounds) * tile;
  return (share + std::min({1.0, share, 0.3 + last})) * tile;
}

// Problems with many rows and a long reduction take the candidate with the shortest expected time instead of the first of
// the library's ranking, where it promises 8 % or more. Over 44 problems with K of 12288 and 13824 the first is 25 % slower
// than the best of 32 on average and up to 2 x, the choice made here 5 %: M=9210 (a 16:9 image being edited beside its
// source, two prompts), N=3072, K=12288 798 -> 493 us; M=6144 682 -> 340. At K = 5120 (66 problems) the first is 7 % off,
// the choice 3 %. Below 8 % the model is as often wrong as right (M=1536, N=3072, K=12288: 4 % promised, 133 -> 141 us
// inside a step); with the margin one of the 110 gets slower. Of two tiles with the same expected time the one that is
// wider in features wins: 256 x 224 takes 244 us at M=4608, 224 x 256 251. With K of 3072 the first is 5 % off, and what
// the model chose instead ran 5 % slower inside a step of 4608 rows, so it stays; below 1024 rows a launch is less than one
// round of large tiles and the model says nothing.
constexpr int kLinRankMinRows = 1024, kLinRankMinK = 4096;
constexpr double kLinRankGain = 0.92, kLinTallTile = 1.01;
constexpr int kLinCandidates = 32;
constexpr size_t kLinTileSums = 256 * 256 * 4;  // what a worker of the kernel passed over leaves of a tile

// The library's kernels for a problem, in its own order, and LinPlan::passed. (All of them at once: a library that has been asked for one alone, and then for
// more of the same problem, has the rest in no order of merit. 0.2 ms, once for a problem.)
static int lin_candidates(hipblasLtHandle_t h, LinPlan& p, size_t lib_ws_bytes, hipblasLtMatmulHeuristicResult_t* res, int* n) {
  hipblasLtMatmulPreference_t pref;
  ODIT_LT(hipblasLtMatmulPreferenceCreate(&pref));
  const uint64_t maxws = lib_ws_bytes;
  hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &maxws, sizeof(maxws));
  *n = 0;
  const hipblasStatus_t st = hipblasLtMatmulAlgoGetHeuristic(h, p.desc, p.a, p.b, p.c, p.d, pref, kLinCandidates, res, n);
  hipblasLtMatmulPreferenceDestroy(pref);
  if (st != HIPBLAS_STATUS_SUCCESS || *n < 1) {
    set_error("odit_linear: hipBLASLt has no kernel for this problem (status %d)", static_cast<int>(st));
    return ODIT_ENOTSUP;
  }
  p.passed = lin_sound(h, res[0].algo) ? 0 : res[0].workspaceSize == 0 ? 1 : 1 + static_cast<int>((res[0].workspaceSize + kLinTileSums - 1) / kLinTileSums);
  return ODIT_OK;
}

static int lin_default_algo(hipblasLtHandle_t h, LinPlan& p, const LinCall& c, size_t lib_ws_bytes) {
  const bool rank = c.M >= kLinRankMinRows && c.K >= kLinRankMinK && c.dtype != ODIT_F32 && !c.first;
  hipblasLtMatmulHeuristicResult_t res[kLinCandidates];
  int n = 0;
  const int rc = lin_candidates(h, p, lib_ws_bytes, res, &n);
  if (rc != ODIT_OK) return rc;
  // What may run; and where the kernel passed over asks for no workspace, as it splits no tile, what asks for none either, if there is any: the
  // same order of summation, and the same bits.
  auto keep = [&](auto wanted) {
    const int m = static_cast<int>(std::stable_partition(res, res + n, wanted) - res);
    if (m > 0) n = m;
    return m > 0;
  };
  if (!keep([&](hipblasLtMatmulHeuristicResult_t& r) { return lin_sound(h, r.algo); })) {
    set_error("odit_linear: hipBLASLt has no kernel for this problem that may be run");
    return ODIT_ENOTSUP;
  }
  if (p.passed == 1) keep([](hipblasLtMatmulHeuristicResult_t& r) { return r.workspaceSize == 0; });
  int best = 0;
  double best_us = 0;  // expected time of the choice, times kLinRankGain for the library's first
  const int cus = rank || p.passed == 1 ? device_cus() : 0;
  for (int i = 0; i < n && cus > 0; ++i) {
    int features, rows;
    bool usual;
    if (res[i].state != HIPBLAS_STATUS_SUCCESS || res[i].workspaceSize > lib_ws_bytes ||
        !lin_macro_tile(hipblaslt_ext::getKernelNameFromAlgo(h, res[i].algo), &features, &rows, &usual)) {
      if (i == 0) break;
      continue;
    }
    const double us = lin_tile_us(c.M, c.N, c.K, features, rows, cus) * (rows > features ? kLinTallTile : 1.);
    if (i == 0) best_us = us * kLinRankGain;
    else if (usual && us < best_us) { best = i; best_us = us; }
  }
  p.algo = res[best].algo;
  p.algo_ws = res[best].workspaceSize;
  p.have_algo = true;
  p.us = static_cast<float>(best == 0 ? best_us / kLinRankGain : best_us);
  return ODIT_OK;
}

// the library's kernel for a plan that has none yet
static int lin_choose_algo(hipblasLtHandle_t h, LinPlan& p, const LinCall& c, size_t lib_ws_bytes) {
  if (p.have_algo && p.algo_ws <= lib_ws_bytes) return ODIT_OK;
  p.tuned = false;  // (what was tuned does not fit into this workspace)
  if (lin_preferred_algo(h, p, c, lib_ws_bytes)) return ODIT_OK;
  return lin_default_algo(h, p, c, lib_ws_bytes);
}

static int lin_check(const LinCall& c) {
  ODIT_CHECK_ARG(c.x && c.w && c.out, "odit_linear: x/w/out must not be null");
  ODIT_CHECK_ARG(c.M >= 0 && c.N > 0 && c.K > 0, "odit_linear: bad shape M=%d N=%d K=%d", c.M, c.N, c.K);
  ODIT_CHECK_ARG(c.dtype == ODIT_BF16 || c.dtype == ODIT_F16 || c.dtype == ODIT_F32, "odit_linear: bad dtype %d", c.dtype);
  ODIT_CHECK_ARG(c.epilogue >= ODIT_EPI_NONE && c.epilogue <= ODIT_EPI_GATED_RESIDUAL_PRE,
                 "odit_linear: unknown epilogue %d", c.epilogue);
  ODIT_CHECK_ARG((c.epilogue != ODIT_EPI_NONE && c.epilogue != ODIT_EPI_GELU_TANH) || c.bias == nullptr,
                 "odit_linear: this epilogue takes no bias");
  ODIT_CHECK_ARG(c.ldx >= c.K && c.ldw >= c.K && c.ldo >= c.N, "odit_linear: leading dimensions too small");
  if (c.epilogue == ODIT_EPI_BIAS || c.epilogue == ODIT_EPI_BIAS_GELU_TANH)
    ODIT_CHECK_ARG(c.bias != nullptr, "odit_linear: this epilogue needs a bias vector");
  if (lin_is_residual(c))
    ODIT_CHECK_ARG(c.residual != nullptr && c.ldr >= c.N, "odit_linear: this epilogue needs `residual` with ldr >= N");
  if (lin_needs_prep(c)) {
    ODIT_CHECK_ARG(c.ws != nullptr, "odit_linear: a gate in the tensor dtype needs a workspace for two fp32 vectors");
    ODIT_CHECK_ARG(c.gate_dtype == c.dtype || c.gate_dtype == ODIT_F32, "odit_linear: gate dtype must equal dtype or be f32");
    ODIT_CHECK_ARG((reinterpret_cast<uintptr_t>(c.ws) & 255) == 0, "odit_linear: workspace must be 256-byte aligned");
  }
  if (c.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE)
    ODIT_CHECK_ARG(c.gate != nullptr && aligned16(c.gate) && aligned16(c.bias),
                   "odit_linear: the pre-scaled form needs a 16-byte aligned float32 gate (and gate*bias) vector");
  return ODIT_OK;
}

}  // namespace odit

// Workspace split: a workspace large enough starts with the hand-written kernel's scratch (tile
// counters that are zero between calls, partial-tile slots); the rest is the library's.
static void lin_split_ws(void* ws, size_t bytes, void** sk, void** lib, size_t* lib_bytes) {
  if (ws != nullptr && bytes >= odit::kGemmScratchBytes + (static_cast<size_t>(1) << 20)) {
    *sk = ws;
    *lib = static_cast<char*>(ws) + odit::kGemmScratchBytes;
    *lib_bytes = bytes - odit::kGemmScratchBytes;
  } else {
    *sk = nullptr;
    *lib = ws;
    *lib_bytes = bytes;
  }
}

static int lin_run_library(const odit::LinCall& c) {
  using namespace odit;
  hipblasLtHandle_t h;
  LinPlan* p;
  const void *alpha, *cptr;
  void* lws;
  size_t lws_bytes;
  int rc = lin_prepare(c, &h, &p, &alpha, &cptr, &lws, &lws_bytes);
  if (rc != ODIT_OK) return rc;
  rc = lin_choose_algo(h, *p, c, lws_bytes);
  if (rc != ODIT_OK) return rc;
  const float beta = lin_is_residual(c) ? 1.f : 0.f;
  ODIT_LT(hipblasLtMatmul(h, p->desc, alpha, c.w, p->a, c.x, p->b, &beta, cptr, p->c, c.out, p->d, &p->algo, lws,
                          lws_bytes, c.stream));
  return ODIT_OK;
}

static odit::GemmCall lin_gemm_call(const odit::LinCall& c, int rows_per_gate, int64_t ldg) {
  odit::GemmCall g;
  g.x = c.x; g.w = c.w; g.bias = c.bias; g.residual = c.residual; g.gate = c.gate; g.out = c.out;
  g.M = c.M; g.N = c.N; g.K = c.K;
  g.ldx = c.ldx; g.ldw = c.ldw; g.ldo = c.ldo; g.ldr = c.ldr;
  g.epilogue = c.epilogue;
  g.gate_f32 = c.gate_dtype == ODIT_F32 ? 1 : 0;
  g.rows_per_gate = rows_per_gate;
  g.ldg = ldg;
  g.clip = c.clip ? 1 : 0;
  return g;
}

// key of the whole problem for the record of what a tuning run found
static odit::LinKey lin_tuned_key(int dev, const odit::LinCall& c, int rows_per_gate, const void* sk) {
  return odit::LinKey{dev, c.M, c.N, c.K, c.epilogue * 4 + (c.bias != nullptr ? 1 : 0) + (c.gate != nullptr ? 2 : 0) + (sk != nullptr ? 0x100 : 0),
                      c.dtype, rows_per_gate, c.ldx, c.ldw, c.ldo};
}

// Which hand-written kernel takes a problem where one is asked for: 1 = the stream-K kernel (few rows; needs its scratch), 2 =
// the tile kernel (many rows), 0 = neither.
constexpr int kTileMinRows = 1025;
static int lin_handwritten_kind(const odit::GemmCall& g, int dtype, const void* sk) {
  if (g.M >= kTileMinRows) return odit::gemm_tile_takes(g, dtype) ? 2 : 0;
  return sk != nullptr && odit::gemm_streamk_takes(g, dtype) ? 1 : 0;
}

static int lin_launch_handwritten(int kind, const odit::GemmCall& g, int dtype, void* sk, hipStream_t stream, int workers = 0) {
  if (kind == 1) return odit::launch_gemm_streamk(&g, 1, dtype, sk, stream);
  if (kind == 3) return odit::launch_gemm_small(&g, 1, dtype, stream);
  if (kind == 4) {
    const odit::TileShares shares = odit::tile_shares(g.M, g.N, g.K, workers);
    if (shares.known && sk != nullptr) return odit::launch_gemm_tile_shared(g, dtype, shares, sk, stream);
    return odit::launch_gemm_tile_apart(g, dtype, stream);
  }
  return odit::launch_gemm_tile(&g, 1, nullptr, dtype, sk, stream);
}

// Whether a hand-written kernel (1 stream-K, 2 tile, 3 small) takes a problem, with this scratch or none.
static bool lin_kind_takes(int kind, const odit::GemmCall& g, int dtype, const void* sk) {
  if (kind == 2) return odit::gemm_tile_takes(g, dtype);
  return (kind == 3 || sk != nullptr) && odit::gemm_streamk_takes(g, dtype);
}

// Whether this thread's plans of the launches that the library makes for a problem hold the kernels that a tuning call chose.
static bool lin_library_tuned(int dev, const odit::LinCall& c, const odit::GemmCall& g) {
  using namespace odit;
  auto tuned = [&](int M) {
    LinCall one = c;
    one.M = M;
    const auto it = g_lin.plans.find(lin_plan_key(dev, one));
    return it != g_lin.plans.end() && it->second.tuned;
  };
  if (g.rows_per_gate <= 0) return tuned(g.M);
  return tuned(g.rows_per_gate) && (g.M % g.rows_per_gate == 0 || tuned(g.M % g.rows_per_gate));
}

// What a tuning call found for a problem, where it holds here: a hand-written kernel has to take these operands (their alignment
// is not in the key), and what the library won with has to be in this thread's plans; the library's own choice, which is what another
// thread would get, may be slower than the kernel that the library's best was measured against.
static bool lin_tuned(int dev, const odit::LinCall& c, const odit::GemmCall& g, const void* sk, odit::Tuned* found) {
  {
    std::lock_guard<std::mutex> lock(odit::g_engine_mu);
    const auto it = odit::g_tuned.find(lin_tuned_key(dev, c, g.rows_per_gate, sk));
    if (it == odit::g_tuned.end()) return false;
    *found = it->second;
  }
  return found->kind == 0 ? lin_library_tuned(dev, c, g) : lin_kind_takes(found->kind, g, c.dtype, sk);
}

// Expected time (us) of one of the library's launches: that of its ranked kernel where it ranks them (long reductions), else 1.29
// PFLOP/s behind 17 us; a long reduction takes 22 us more where it is split over few output tiles. Fitted to the launches that
// the tile kernel's time is fitted to (11 %). Choosing by the two expected times takes 1 % longer over them than the better of
// both would, the library alone 5 %.
static float lin_library_us(const odit::LinCall& c, int M) {
  using namespace odit;
  if (M >= kLinRankMinRows && c.K >= kLinRankMinK && c.dtype != ODIT_F32) {
    LinCall one = c;
    one.M = M;
    hipblasLtHandle_t h;
    LinPlan* p;
    const size_t gb = lin_gate_bytes(one);
    if (gb <= one.ws_bytes && lin_find_plan(one, &h, &p) == ODIT_OK && lin_choose_algo(h, *p, one, one.ws ? one.ws_bytes - gb : 0) == ODIT_OK && p->us > 0)
      return p->us;
  }
  const float us = 16.6f + 2e-9f * M * c.N * c.K / 1.286f;
  return c.K >= 2 * c.N && static_cast<int64_t>(M) * c.N < 128 * 65536 ? us + 22.f : us;
}
static float lin_library_us(const odit::LinCall& c, const odit::GemmCall& g) {  // (a launch for each group of rows with a gate vector of its own)
  if (g.rows_per_gate <= 0) return lin_library_us(c, g.M);
  const int full = g.M / g.rows_per_gate, last = g.M % g.rows_per_gate;
  return full * lin_library_us(c, g.rows_per_gate) + (last > 0 ? lin_library_us(c, last) : 0.f);
}

// Whether the library's first choice for a problem (of launches for groups of rows, the first group's) is one that never runs: LinPlan::passed.
static int lin_passed(const odit::LinCall& c, const odit::GemmCall& g) {
  using namespace odit;
  LinCall one = c;
  if (g.rows_per_gate > 0) one.M = g.rows_per_gate;
  hipblasLtHandle_t h;
  LinPlan* p;
  const size_t gb = lin_gate_bytes(one), room = one.ws && gb <= one.ws_bytes ? one.ws_bytes - gb : 0;
  if (lin_find_plan(one, &h, &p) != ODIT_OK || p->tuned) return 0;  // (the call says what is wrong)
  if (p->passed != 0 || p->have_algo) return p->passed;
  hipblasLtMatmulHeuristicResult_t res[kLinCandidates];
  int n = 0;
  return lin_preferred_algo(h, *p, one, room) || lin_candidates(h, *p, room, res, &n) != ODIT_OK ? 0 : p->passed;
}

// The stream-K kernel for one problem: where the reduction is long against the number of output features (K >= 2 N: the
// library's choices split K badly there: M=80, N=3072, K=12288 57 us against 31, M=512 69 against 52, M=1024 110 against 85) and
// there is work for all CUs; with a small product (kSmallWeights: a few MB of weights) its ranges would be shorter than what
// handing partial tiles over costs (M=256, N=256, K=1024: 19 us against 10).
constexpr int64_t kSmallWeights = 1ll << 22;  // N K
static bool lin_streamk_rule(const odit::GemmCall& g) {
  return g.K >= 2 * g.N && g.M >= 48 && g.M < kTileMinRows && static_cast<int64_t>(g.N) * g.K >= kSmallWeights;
}

// The kernel of a problem that names no engine: what a tuning call found, else the stream-K kernel by its rule or the tile kernel,
// whose expected time is shorter (N=3072, K=12288, us, stream-K / tile: 300 rows 43 / 49, 400 48 / 49, 512 52 / 56, 592 61 / 55, 1024
// 84 / 75; N=5120, K=13824: 200 62 / 60, 300 65 / 60, 592 101 / 86, 1024 144 / 112), else the kernel for small products (3) by its
// rule, else the tile kernel where its expected time is below the library's (kTileMinAuto rows or more), else the library (0). One
// launch of the library takes 8 to 10 us for any small product, the small kernel 4 to 7 up to K = kSmallK; beside a second
// problem, whose launch it saves, up to kSmallPairK.
constexpr int kSmallK = 1024, kSmallPairK = 2048;
constexpr int kTileMinAuto = 256;

// What a tuning call times against the library: every kernel that the rules may choose for the problem (one problem alone or half
// of a pair, so that no tuned problem is left with less than it had), and the tile kernel for few rows too.
static bool lin_candidate(int kind, const odit::GemmCall& g, int dtype, const void* sk) {
  if (!lin_kind_takes(kind, g, dtype, sk)) return false;
  if (kind == 1) return g.M < kTileMinRows;
  return kind == 2 || odit::gemm_small_rule(&g, 1, odit::device_cus(), kSmallPairK);
}

// Time of a problem's own call: the better of what it may run on, by expectation, or what a tuning call measured where that is
// shorter. (It is behind a flush often 5 to 10 us longer than in a model: taken for itself it made two calls look slower than they
// are, and 1122 + 185 rows, N=12288, K=3072, 103 us in two calls, went to one launch of 106.)
static float lin_call_us(int dev, const odit::LinCall& c, const odit::GemmCall& g, const void* sk) {
  const bool scratch = sk != nullptr;
  float us = lin_library_us(c, g);
  const int cus = odit::device_cus();
  if (scratch && lin_streamk_rule(g) && odit::gemm_streamk_takes(g, c.dtype)) {
    const float own = odit::gemm_streamk_us(g.M, 0, g.N, g.K, cus);
    if (own > 0.f && own < us) us = own;
  }
  if (g.M >= kTileMinAuto && odit::gemm_tile_takes(g, c.dtype)) {
    const odit::TilePlan plan = odit::plan_gemm_tile(&g, 1, cus, scratch);
    if (plan.bm > 0 && plan.us < us) us = plan.us;
  }
  odit::Tuned found;
  if (lin_tuned(dev, c, g, sk, &found) && found.us < us) us = found.us;
  return us;
}
static int lin_rule_kind(const odit::LinCall& c, const odit::GemmCall& g, const void* sk) {
  const bool takes = g.M >= kTileMinAuto && odit::gemm_tile_takes(g, c.dtype), tile = !c.no_tile && takes;
  if (sk != nullptr && lin_streamk_rule(g) && odit::gemm_streamk_takes(g, c.dtype)) {
    const int cus = odit::device_cus();
    const odit::TilePlan plan = tile ? odit::plan_gemm_tile(&g, 1, cus, true) : odit::TilePlan{};
    return plan.bm > 0 && plan.us < odit::gemm_streamk_us(g.M, 0, g.N, g.K, cus) ? 2 : 1;
  }
  if (!c.no_tile && odit::gemm_streamk_takes(g, c.dtype) && odit::gemm_small_rule(&g, 1, odit::device_cus(), kSmallK)) return 3;
  if (!takes) return 0;
  const odit::TilePlan plan = odit::plan_gemm_tile(&g, 1, odit::device_cus(), sk != nullptr);
  if (plan.bm == 0) return 0;
  if (tile && plan.us < lin_library_us(c, g)) return 2;
  // In the place of a kernel that never runs the tile kernel does. A call that wants no other order of summation has every tile whole where that kernel would have had it so,
  // and the library's order of operations in the epilogue (kind 4): the library's bits. (65520 rows of a pair, us, the library's next / this: N=15360, K=5120 7690 / 6930,
  // N=5120 gated 2750 / 2340, K=13824 7200 / 6010. The library's next kernel without a workspace, of another tile, can differ: N=15360 with GELU, 2875 rows.) Where it would have split tiles
  // this kernel parts the same ones there (gemm_tile_shared.hip; us, bf16, that kernel / this: 13202 rows, N=15360, K=5120 1519 / 1642, N=13824 with GELU 1640 / 1554,
  // N=5120, K=13824 1513 / 1547; 8192 rows, N=9216, K=3072 449 / 373; 34968 rows, N=15360, K=5120 3911 / 4396; 2400 rows, N=5120, K=13824, fewer tiles than
  // workers, 436 / 278).
  const int passed = lin_passed(c, g);
  return passed == 0 ? 0 : tile ? 2 : 4;
}
// for kind 4: how many workers the kernel passed over would have shared tiles out among (0: none is)
static int lin_workers(const odit::LinCall& c, const odit::GemmCall& g) { return std::max(lin_passed(c, g) - 1, 0); }
static int lin_auto_kind(int dev, const odit::LinCall& c, const odit::GemmCall& g, const void* sk) {
  odit::Tuned found;
  return lin_tuned(dev, c, g, sk, &found) ? found.kind : lin_rule_kind(c, g, sk);
}

int odit::linear_tile_unless(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int dtype, void* workspace,
                             size_t workspace_bytes, const int* unless, bool ask, hipStream_t stream) {
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  const LinCall c{x, w, bias, nullptr, nullptr, out, M, N, K, K, ldw, N, 0, bias != nullptr ? ODIT_EPI_BIAS : ODIT_EPI_NONE, dtype, dtype, lib, lib_bytes, stream};
  const int rc = lin_check(c);
  if (rc != ODIT_OK) return rc;
  const GemmCall g = lin_gemm_call(c, 0, 0);
  int dev = 0;
  if (M < kTileMinAuto || !gemm_tile_takes(g, dtype) || hipGetDevice(&dev) != hipSuccess) return ODIT_ENOTSUP;
  // a launch that mostly ends at once may be behind the best one by a little where it does not
  const TilePlan plan = plan_gemm_tile(&g, 1, device_cus(), sk != nullptr);
  if (plan.bm == 0 || plan.us > 1.15f * lin_call_us(dev, c, g, sk)) return ODIT_ENOTSUP;
  return ask ? ODIT_OK : launch_gemm_tile_unless(g, unless, dtype, sk, stream);
}

// whether ODIT_LINEAR_CLIP (`bit`) asks anything of a call
static bool lin_clips(const odit::LinCall& c, unsigned flags, unsigned bit) { return (flags & bit) != 0 && c.dtype == ODIT_F16 && odit::lin_is_residual(c); }

// a clip of what the library has written: eight values to a thread where the rows' starts allow (`wide`)
__global__ __launch_bounds__(256) void lin_clip_kernel(odit::f16_t* out, int M, int N, int64_t ldo, int wide) {
  for (int row = blockIdx.x; row < M; row += gridDim.x) {
    odit::f16_t* const at = out + row * ldo;
    for (int col = 8 * static_cast<int>(threadIdx.x); col < N; col += 8 * 256) {
      if (wide) {
        odit::u32x4* const v = reinterpret_cast<odit::u32x4*>(at + col);
        odit::u32x4 o = *v;
#pragma unroll
        for (int p = 0; p < 4; ++p) odit::Raw<odit::f16_t>::set2(o, p, odit::f16_clipped(odit::Raw<odit::f16_t>::get(o, 2 * p)), odit::f16_clipped(odit::Raw<odit::f16_t>::get(o, 2 * p + 1)));
        *v = o;
      } else {
        for (int u = col; u < N && u < col + 8; ++u) at[u] = odit::from_float<odit::f16_t>(odit::f16_clipped(odit::to_float(at[u])));
      }
    }
  }
}
static int lin_clip(const odit::LinCall& c) {
  const int wide = c.N % 8 == 0 && c.ldo % 8 == 0 && odit::aligned16(c.out) ? 1 : 0;
  hipLaunchKernelGGL(lin_clip_kernel, dim3(static_cast<unsigned>(c.M)), dim3(256), 0, c.stream, static_cast<odit::f16_t*>(c.out), c.M, c.N, c.ldo, wide);
  return odit::check_launch("odit_linear (clip)");
}

extern "C" int odit_linear_prefer(int M, int N, int K, int dtype, int solution) {
  using namespace odit;
  ODIT_CHECK_ARG(M > 0 && N > 0 && K > 0 && solution >= 0, "odit_linear_prefer: bad problem or solution index");
  std::lock_guard<std::mutex> lock(g_engine_mu);
  for (Preferred& e : g_preferred)
    if (e.m == M && e.n == N && e.k == K && e.dtype == dtype) { e.solution = solution; return ODIT_OK; }
  if (g_preferred.size() >= 1024) { set_error("odit_linear_prefer: more than 1024 problems"); return ODIT_EINVAL; }
  g_preferred.push_back({M, N, K, dtype, solution});
  return ODIT_OK;
}

extern "C" size_t odit_linear_workspace_bytes(void) {
  return odit::kGemmScratchBytes + (static_cast<size_t>(64) << 20);
}

extern "C" int odit_linear_rows(const void* x, const void* w, const void* bias, void* out, const void* residual,
                                const void* gate, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                int64_t ldr, int epilogue, int gate_dtype, int dtype, int rows_per_gate,
                                int64_t gate_stride, unsigned flags, void* workspace, size_t workspace_bytes,
                                void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG((flags & ~(ODIT_LINEAR_LIBRARY | ODIT_LINEAR_HANDWRITTEN | ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE | ODIT_LINEAR_CLIP)) == 0 &&
                     (flags & (ODIT_LINEAR_LIBRARY | ODIT_LINEAR_HANDWRITTEN)) != (ODIT_LINEAR_LIBRARY | ODIT_LINEAR_HANDWRITTEN),
                 "odit_linear_rows: flags may name one engine (ODIT_LINEAR_LIBRARY or ODIT_LINEAR_HANDWRITTEN), ODIT_LINEAR_FIRST, ODIT_LINEAR_NO_TILE and ODIT_LINEAR_CLIP, got %#x", flags);
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  LinCall c{x, w, bias, residual, gate, out, M, N, K, ldx, ldw, ldo, ldr, epilogue, gate_dtype, dtype,
            lib, lib_bytes, static_cast<hipStream_t>(stream)};
  c.first = (flags & ODIT_LINEAR_FIRST) != 0;
  c.no_tile = c.first || (flags & ODIT_LINEAR_NO_TILE) != 0;
  int rc = lin_check(c);
  if (rc != ODIT_OK || M == 0) return rc;
  c.clip = lin_clips(c, flags, ODIT_LINEAR_CLIP);
  ODIT_CHECK_ARG(rows_per_gate >= 0 && (rows_per_gate == 0 || gate_stride >= 0),
                 "odit_linear_rows: rows_per_gate and gate_stride must not be negative");
  const bool per_rows = lin_is_residual(c) && gate != nullptr && rows_per_gate > 0 && rows_per_gate < M;
  const int engine = lin_engine_of(flags);
  const GemmCall g = lin_gemm_call(c, per_rows ? rows_per_gate : 0, per_rows ? gate_stride : 0);
  int dev = 0, kind = 0;
  if (engine == 2) {
    kind = lin_handwritten_kind(g, dtype, sk);
    if (kind == 0) {
      set_error("odit_linear: no hand-written kernel takes this problem (M=%d N=%d K=%d, workspace %zu bytes)",
                M, N, K, workspace_bytes);
      return ODIT_ENOTSUP;
    }
  } else if (engine == 0 && hipGetDevice(&dev) == hipSuccess) {
    kind = lin_auto_kind(dev, c, g, sk);
  }
  const int workers = kind == 4 ? lin_workers(c, g) : 0;
  const bool apart = per_rows && workers > 0;
  if (kind != 0 && !apart) return lin_launch_handwritten(kind, g, dtype, sk, c.stream, workers);
  if (!per_rows) {
    rc = lin_run_library(c);
    return rc == ODIT_OK && c.clip ? lin_clip(c) : rc;
  }
  // the library's epilogue takes one gate vector per launch: one launch per group of rows (`apart`: and which tiles are split follows from a group's)
  const size_t esz = dtype == ODIT_F32 ? 4 : 2, gsz = gate_dtype == ODIT_F32 ? 4 : esz;
  for (int r0 = 0; r0 < M; r0 += rows_per_gate) {
    LinCall cg = c;
    const int64_t grp = r0 / rows_per_gate;
    cg.M = M - r0 < rows_per_gate ? M - r0 : rows_per_gate;
    cg.x = static_cast<const char*>(x) + static_cast<size_t>(r0) * ldx * esz;
    cg.out = static_cast<char*>(out) + static_cast<size_t>(r0) * ldo * esz;
    cg.residual = static_cast<const char*>(residual) + static_cast<size_t>(r0) * ldr * esz;
    cg.gate = static_cast<const char*>(gate) + static_cast<size_t>(grp * gate_stride) * gsz;
    if (epilogue == ODIT_EPI_GATED_RESIDUAL_PRE && bias != nullptr)
      cg.bias = static_cast<const char*>(bias) + static_cast<size_t>(grp * gate_stride) * 4;
    const GemmCall gg = lin_gemm_call(cg, 0, 0);
    if (apart && lin_rule_kind(cg, gg, sk) == 4) rc = lin_launch_handwritten(4, gg, dtype, sk, c.stream, lin_workers(cg, gg));
    else rc = lin_run_library(cg);
    if (rc != ODIT_OK) return rc;
  }
  return c.clip ? lin_clip(c) : ODIT_OK;
}

// Two problems in one launch, or two calls? By expected time, or what was measured for a tuned problem if that is shorter (811
// + 466 rows, N=9216, K=3072: 73 us in one launch, 93 in two tuned calls; 1216 + 448, N=6144, K=1024: 30 and 36). One launch has
// one set of overheads for both, shares the tiles of the last round out over all CUs and takes gates that differ per batch
// entry, for which the library needs a call per entry.
// Measured at width 3072 (us, stream-K pair / tile kernel pair / two calls): 512 + 80 QKV 47 / 55 / 71, MLP up 61 / 58 / 70, out 29 /
// 28 / 37, MLP down 67 / 61 / 90; 810 + 466 QKV 97 / 69 / 84, out 45 / 40 / 44, up 131 / 103 / 107, down 116 / 101 / 126; 3024 + 642 QKV -
// / 169 / 183, out - / 65 / 83, up - / 219 / 241, down - / 231 / 246. The stream-K kernel's fit ends at kPairTiles tiles of 128 rows
// together, kPairTilesGated where the library would need a call per entry: past them only the tile kernel is compared.
// Two calls are put 3 % above the sum of their estimates (the second one's rows and weights are cold when it starts). Over 104
// pairs of 267 to 8759 and 40 to 885 rows, all four products of a dual-stream block (ms): 15.30 by this margin, 15.27 by the better of
// the three each time, 15.33 with 0 or 6 % in the place of the 3, 15.70 where the tile kernel had to promise 6 %. (Measured with the times that one
// problem's form has; plan_streamk says what a pair's cost by now.)
constexpr int kPairTiles = 8, kPairTilesGated = 20;
constexpr float kPairGain = 1.03f;

extern "C" int odit_linear_pair(const odit_linear_problem* q, int N, int K, int epilogue, int gate_dtype, int dtype, unsigned flags,
                                void* workspace, size_t workspace_bytes, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(q != nullptr, "odit_linear_pair: null problems");
  const int engine = lin_engine_of(flags);
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  GemmCall g[2];
  bool per_rows = false, takes = true, streamk = sk != nullptr && engine != 1;
  bool tile = engine != 1 && (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) == 0;
  int tiles = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { set_error("odit_linear_pair: hipGetDevice failed"); return ODIT_ELAUNCH; }
  LinCall calls[2];
  for (int i = 0; i < 2; ++i) {
    const LinCall& c = calls[i] = LinCall{q[i].x, q[i].w, q[i].bias, q[i].residual, q[i].gate, q[i].out, q[i].M, N, K, q[i].ldx, q[i].ldw, q[i].ldo, q[i].ldr,
                    epilogue, gate_dtype, dtype, lib, lib_bytes, static_cast<hipStream_t>(stream)};
    const int rc = lin_check(c);
    if (rc != ODIT_OK) return rc;
    ODIT_CHECK_ARG(q[i].rows_per_gate >= 0 && q[i].gate_stride >= 0, "odit_linear_pair: rows_per_gate and gate_stride must not be negative");
    const bool rows = lin_is_residual(c) && q[i].gate != nullptr && q[i].rows_per_gate > 0 && q[i].rows_per_gate < q[i].M;
    calls[i].clip = lin_clips(c, flags, i == 0 ? ODIT_LINEAR_CLIP : ODIT_LINEAR_CLIP2);
    g[i] = lin_gemm_call(c, rows ? q[i].rows_per_gate : 0, rows ? q[i].gate_stride : 0);
    per_rows = per_rows || rows;
    takes = takes && q[i].M > 0 && gemm_streamk_takes(g[i], dtype);
    streamk = streamk && takes;
    tile = tile && q[i].M > 0 && gemm_tile_takes(g[i], dtype);
    if (engine == 1 || (!takes && !tile)) return ODIT_ENOTSUP;
    tiles += (q[i].M + kGemmBM - 1) / kGemmBM;
  }
  const int cus = device_cus();
  if (engine == 2) return streamk ? launch_gemm_streamk(g, 2, dtype, sk, static_cast<hipStream_t>(stream)) : ODIT_ENOTSUP;
  if (static_cast<int64_t>(N) * K < (1 << 14)) return ODIT_ENOTSUP;
  if (takes && (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) == 0 && engine == 0 && gemm_small_rule(g, 2, cus, kSmallPairK))
    return launch_gemm_small(g, 2, dtype, static_cast<hipStream_t>(stream));
  // (no message where the answer is ODIT_ENOTSUP: two calls are an ordinary answer)
  const bool small = streamk && tiles <= (per_rows ? kPairTilesGated : kPairTiles);
  const TilePlan plan = tile ? plan_gemm_tile(g, 2, cus, sk != nullptr) : TilePlan{};
  const bool wide = plan.bm > 0 && plan.us < kPairGain * (lin_call_us(dev, calls[0], g[0], sk) + lin_call_us(dev, calls[1], g[1], sk));
  if (small && !(wide && plan.us < gemm_streamk_us(g[0].M, g[1].M, N, K, cus)))
    return launch_gemm_streamk(g, 2, dtype, sk, static_cast<hipStream_t>(stream));
  if (!wide) return ODIT_ENOTSUP;
  return launch_gemm_tile(g, 2, nullptr, dtype, sk, static_cast<hipStream_t>(stream));
}

extern "C" int odit_linear_pair_is_small(int M0, int M1, int N, int K) {
  using namespace odit;
  if (M0 <= 0 || M1 <= 0 || N <= 0 || K <= 0 || K % kGemmBK != 0 || N % 8 != 0 || static_cast<int64_t>(N) * K < (1 << 14)) return 0;
  GemmCall g[2] = {};
  for (int i = 0; i < 2; ++i) { g[i].M = i == 0 ? M0 : M1; g[i].N = N; g[i].K = K; }
  const int cus = device_cus();
  return cus > 0 && gemm_small_rule(g, 2, cus, kSmallPairK) ? 1 : 0;
}

// Two projections that read the same rows, in one launch of the tile kernel or two calls, by expected time (2 % have to be
// promised: where two calls would run this kernel too, its estimate is off by the same for both). What one launch
// gains is full rounds (M=1536, N=9216 and 12288, K=3072: 504 tiles, 1.97 rounds, 150 us; 216 and 288 in two calls 194) and the
// rows' pieces in L2 for both.
constexpr float kOneLaunchGain = .98f;

// The same for a third one, of other rows (what it is compared with: the first one's call and the others in one launch or two calls).
// Wan's QKV with the cross-attention's keys and values, whose rows are there from the start, us, apart / one launch: 2706 rows and 512 353 +
// 60 / 364; 5000 and 512 584 + 60 / 601; 2048 and 512 238 + 60 / 287; 1500 and 512 188 + 60 / 244.
static int lin_beside(const char* name, const odit_linear_problem* q, int count, const int* N, int K, const int* epilogue, int dtype, unsigned flags,
                      int launch, bool force, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace odit;
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { set_error("%s: hipGetDevice failed", name); return ODIT_ELAUNCH; }
  GemmCall g[3];
  const bool tile = (lin_engine_of(flags) == 0 || force) && (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) == 0;
  const bool choose = !force && launch != ODIT_LAUNCH_ANSWERED;
  float us[3] = {0.f, 0.f, 0.f};
  for (int i = 0; i < count; ++i) {
    const LinCall c{q[i].x, q[i].w, q[i].bias, nullptr, nullptr, q[i].out, q[i].M, N[i], K, q[i].ldx, q[i].ldw, q[i].ldo, 0,
                    epilogue[i], dtype, dtype, lib, lib_bytes, static_cast<hipStream_t>(stream)};
    const int rc = lin_check(c);
    if (rc != ODIT_OK) return rc;
    if (lin_is_residual(c)) { set_error("%s: no residual", name); return ODIT_EINVAL; }
    g[i] = lin_gemm_call(c, 0, 0);
    if (!tile || (!force && q[i].M < kTileMinAuto) || !gemm_tile_takes(g[i], dtype)) return ODIT_ENOTSUP;
    if (choose) us[i] = lin_call_us(dev, c, g[i], sk);
  }
  const int cus = device_cus();
  const TilePlan plan = plan_gemm_tile(g, count, cus, sk != nullptr);
  if (plan.bm == 0) return ODIT_ENOTSUP;
  if (choose) {
    float others = us[1] + us[2];
    if (count == 3) {
      const TilePlan two = plan_gemm_tile(g + 1, 2, cus, sk != nullptr);
      if (two.bm > 0 && two.us < others) others = two.us;
    }
    if (plan.us >= kOneLaunchGain * (us[0] + others)) return ODIT_ENOTSUP;
  }
  return launch == ODIT_LAUNCH_ASK ? ODIT_OK : launch_gemm_tile(g, count, nullptr, dtype, sk, static_cast<hipStream_t>(stream));
}

extern "C" int odit_linear_fork(const odit_linear_problem* q, const int* N, int K, const int* epilogue, int dtype, unsigned flags, void* workspace,
                                size_t workspace_bytes, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(q != nullptr && N != nullptr && epilogue != nullptr, "odit_linear_fork: null arguments");
  return lin_beside("odit_linear_fork", q, 2, N, K, epilogue, dtype, flags, ODIT_LAUNCH_CHOOSE, false, workspace, workspace_bytes, stream);
}

extern "C" int odit_linear_three(const odit_linear_problem* q, const int* N, int K, const int* epilogue, int dtype, unsigned flags, int launch,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(q != nullptr && N != nullptr && epilogue != nullptr, "odit_linear_three: null arguments");
  return lin_beside("odit_linear_three", q, 3, N, K, epilogue, dtype, flags, launch, lin_engine_of(flags) == 2, workspace, workspace_bytes, stream);
}

// Projections to query, key and value heads with the heads' norm and rotation at the tile's end, or the projections and a pass over
// their output, by expected time. The pass takes 6 us and 8 bytes for every feature of q at 5 TB/s; the tile's end 4.5 us more a round
// on 256-row tiles and 1.3 on 128-row ones (its arithmetic has no matrix work to hide behind). Beside a projection without heads nothing is
// counted for it: a GELU tile's end is as long, and where the other has no GELU, as much is gained that is not counted either (charged for
// the rounds of the heads' tiles, 19 of 2160 answers change, every one to the slower way. us with cold weights, apart / one launch: K=512, 2500
// rows, N=6144 beside 4 heads of 64 53.0 / 48.2, 1800 rows, N=6144 beside 8 of 128 50.9 / 48.0; K=1024, 3000 rows, N=9216 beside 24 of 128
// 155 / 138). What would be one launch of the tile kernel anyway nearly always takes the pass with it. Kernel time in a
// model, us, projections + pass / one launch: 2048 + 342 rows, N=9216, K=3072 119 + 17 / 130; 1024 + 512 rows 73 + 11 / 79; 8192 + 512
// rows 340 + 45 / 365; 1536 rows, N=12288 with GELU beside N=9216 153 + 10 / 157; 4608 rows 435 + 25 / 438. Few rows, where the
// stream-K kernel takes the pair, stay there unless the tile kernel wins with its time of cold weights (kColdTile times the
// expected one, which is of a round in which others fetch the same): 512 + 80 rows 48 + 6 / 56, in the model 0.5 % slower. The same
// holds for rows that would take two calls otherwise: 772 rows, N=9216 beside N=12288 with GELU 52 + 64 + 7 / 129.
constexpr float kColdTile = 1.18f;

// (rows or features that do not fit the heads: false, with the message set)
static bool lin_heads_out(const char* name, const odit_linear_problem& q, int N, const odit_head_output& o, odit::HeadsOut* h) {
  if (!(o.S > 0 && o.H > 0 && o.D > 0 && o.offset >= 0 && o.offset + static_cast<int64_t>(o.S) <= o.S_total && q.M % o.S == 0 &&
        static_cast<int64_t>(o.H) * o.D * 3 == N && static_cast<int64_t>(q.M / o.S) * o.S_total < (1ll << 31))) {
    odit::set_error("%s: rows or features do not fit the heads", name);
    return false;
  }
  *h = odit::HeadsOut{o.q, o.k, o.v, o.wq, o.wk, o.cos, o.sin, o.S, o.offset, o.S_total, o.H * o.D, o.D, 0, 0, o.eps};
  return true;
}

extern "C" int odit_linear_heads(const odit_linear_problem* q, const int* N, int K, const int* epilogue, const odit_head_output* const* heads, int dtype,
                                 unsigned flags, int launch, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(q != nullptr && N != nullptr && epilogue != nullptr && heads != nullptr && (heads[0] != nullptr || heads[1] != nullptr),
                 "odit_linear_heads: null arguments");
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { set_error("odit_linear_heads: hipGetDevice failed"); return ODIT_ELAUNCH; }
  const int engine = lin_engine_of(flags);
  if (engine == 1 || (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) != 0) return ODIT_ENOTSUP;
  GemmCall g[2];
  HeadsOut h[2];
  LinCall calls[2];
  float apart = 0.f, pass = 6.f;
  bool both = true;
  for (int i = 0; i < 2; ++i) {
    h[i] = HeadsOut{};
    LinCall& c = calls[i] = LinCall{q[i].x, q[i].w, q[i].bias, nullptr, nullptr, q[i].out, q[i].M, N[i], K, q[i].ldx, q[i].ldw, q[i].ldo, 0,
                                    epilogue[i], dtype, dtype, lib, lib_bytes, static_cast<hipStream_t>(stream)};
    if (heads[i] != nullptr) {
      if (!lin_heads_out("odit_linear_heads", q[i], N[i], *heads[i], &h[i])) return ODIT_EINVAL;
      c.out = heads[i]->q;
      c.ldo = N[i];
      pass += 8.f / 15e6f * q[i].M * N[i];
    }
    both = both && heads[i] != nullptr;
    const int rc = lin_check(c);
    if (rc != ODIT_OK) return rc;
    ODIT_CHECK_ARG(!lin_is_residual(c), "odit_linear_heads: no residual");
    g[i] = lin_gemm_call(c, 0, 0);
    if (!gemm_tile_takes(g[i], dtype) || (heads[i] != nullptr && !gemm_tile_heads_takes(g[i], h[i]))) return ODIT_ENOTSUP;
  }
  auto tile = [&] { return launch == ODIT_LAUNCH_ASK ? ODIT_OK : launch_gemm_tile_heads(g, 2, h, dtype, sk, static_cast<hipStream_t>(stream)); };
  if (engine == 2) return tile();
  const int cus = device_cus();
  const bool pair = both && N[0] == N[1], streamk_takes = pair && gemm_streamk_takes(g[0], dtype) && gemm_streamk_takes(g[1], dtype);
  if (streamk_takes && gemm_small_rule(g, 2, cus, kSmallPairK)) {
    if (h[0].D != 64 || h[1].D != 64) return ODIT_ENOTSUP;  // (a tile of the small kernel is a head of 64 features)
    return launch == ODIT_LAUNCH_ASK ? ODIT_OK : launch_gemm_small_heads(g, 2, h, dtype, static_cast<hipStream_t>(stream));
  }
  if (launch == ODIT_LAUNCH_ANSWERED) return tile();
  for (int i = 0; i < 2; ++i) apart += lin_call_us(dev, calls[i], g[i], sk);
  const TilePlan plan = plan_gemm_tile(g, 2, cus, sk != nullptr);
  if (plan.bm == 0) return ODIT_ENOTSUP;
  const int rounds = (plan.tiles + cus - 1) / cus;
  const float end = both ? (plan.bm == 256 ? 4.5f : 1.3f) * rounds : 0.f;
  if (pair) {  // what odit_linear_pair would choose
    apart *= kPairGain;
    const int tiles = (g[0].M + kGemmBM - 1) / kGemmBM + (g[1].M + kGemmBM - 1) / kGemmBM;
    const float streamk = sk != nullptr && streamk_takes && tiles <= kPairTiles ? gemm_streamk_us(g[0].M, g[1].M, N[0], K, cus) : 0.f;
    if (streamk > 0.f && !(plan.us < apart && plan.us < streamk)) apart = streamk - (kColdTile - 1.f) * plan.us;
  } else {
    apart *= kOneLaunchGain;
    if (plan.us >= apart) apart -= (kColdTile - 1.f) * plan.us;
  }
  if (plan.us + end >= (plan.us < apart ? plan.us : apart) + pass) return ODIT_ENOTSUP;
  return tile();
}

// LayerNorm and modulation in front of a pair that the small kernel takes, up to 4 steps of the reduction. us, the norm's launch and the pair's /
// one launch, one after the other without the host: M=256+64, K=256, heads of N=768 6.48 / 5.67, N=1024 with GELU 6.45 / 5.61; M=64+64, K=128,
// N=512 5.76 / 4.35; with 8 steps, M=512+64, K=512, heads of N=1536 8.40 / 9.02 (every workgroup norms its rows again). The host, which such a
// model mostly waits for, is asked for a launch less: 3.6 us. One problem of a longer reduction and few features, a large model's head: linear_head.hip.
static int lin_normed(const char* name, const odit_linear_problem* q, const odit_row_norm* norm, int count, int N, int K, int epilogue,
                      const odit_head_output* const* heads, int dtype, unsigned flags, int launch, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(q != nullptr && norm != nullptr && (heads == nullptr || (heads[0] != nullptr && heads[1] != nullptr)), "%s: null arguments", name);
  if (lin_engine_of(flags) != 0 || (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) != 0) return ODIT_ENOTSUP;
  GemmCall g[2];
  HeadsOut h[2];
  RowNorm r[2];
  for (int i = 0; i < count; ++i) {
    LinCall c{q[i].x, q[i].w, q[i].bias, nullptr, nullptr, q[i].out, q[i].M, N, K, q[i].ldx, q[i].ldw, q[i].ldo, 0, epilogue, dtype, dtype, nullptr, 0,
              static_cast<hipStream_t>(stream)};
    if (heads != nullptr) {
      if (!lin_heads_out(name, q[i], N, *heads[i], &h[i])) return ODIT_EINVAL;
      c.out = heads[i]->q;
      c.ldo = N;
    }
    const int rc = lin_check(c);
    if (rc != ODIT_OK) return rc;
    ODIT_CHECK_ARG(!lin_is_residual(c), "%s: no residual", name);
    const odit_row_norm& n = norm[i];
    ODIT_CHECK_ARG(n.shift != nullptr && n.scale != nullptr && n.S > 0 && n.stride >= 0, "%s: bad modulation rows", name);
    g[i] = lin_gemm_call(c, 0, 0);
    r[i] = RowNorm{n.shift, n.scale, n.stride, n.S, n.eps};
    if (count == 1 && heads == nullptr && K > kSmallNormK) {
      const int features = linear_head_features(g[0], r[0], dtype, device_cus());
      if (features == 0) return ODIT_ENOTSUP;
      return launch == ODIT_LAUNCH_ASK ? ODIT_OK : launch_linear_head(g[0], r[0], features, dtype, static_cast<hipStream_t>(stream));
    }
    if (!aligned16(n.shift) || !aligned16(n.scale) || n.stride % 8 != 0 || K > kSmallNormK || !gemm_streamk_takes(g[i], dtype) ||
        (heads != nullptr && (h[i].D != 64 || !gemm_tile_takes(g[i], dtype) || !gemm_tile_heads_takes(g[i], h[i]))))
      return ODIT_ENOTSUP;
  }
  if (static_cast<int64_t>(N) * K < (1 << 14) || !gemm_small_rule(g, count, device_cus(), kSmallNormK)) return ODIT_ENOTSUP;
  return launch == ODIT_LAUNCH_ASK ? ODIT_OK : launch_gemm_small_norm(g, count, r, heads != nullptr ? h : nullptr, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int odit_linear_pair_norm(const odit_linear_problem* q, const odit_row_norm* norm, int N, int K, int epilogue,
                                     const odit_head_output* const* heads, int dtype, unsigned flags, int launch, void* stream) {
  return lin_normed("odit_linear_pair_norm", q, norm, 2, N, K, epilogue, heads, dtype, flags, launch, stream);
}

extern "C" int odit_linear_norm(const odit_linear_problem* q, const odit_row_norm* norm, int N, int K, int epilogue, int dtype, unsigned flags, void* stream) {
  return lin_normed("odit_linear_norm", q, norm, 1, N, K, epilogue, nullptr, dtype, flags, ODIT_LAUNCH_ANSWERED, stream);
}

// What a small model's step begins with: two projections that hang on nothing but the inputs, with the norm of one of them. us, three
// launches one after the other / one: 256 rows of 64 and 64 rows of 256 to 256 features 9.7 / 4.75, 1024 and 128 rows 9.9 / 4.8, 64 rows of 64 and 20 of 128
// to 128 8.3 / 3.6. And what it ends with (odit_linear_norm), norm and projection: 256 rows of 256 to 64 features 7.4 / 5.3, 2 x 512 7.5 / 5.3.
extern "C" int odit_linear_stem(const odit_linear_problem* q, int N, const int K[2], const void* weight, float eps, int dtype, unsigned flags, void* stream) {
  using namespace odit;
  ODIT_CHECK_ARG(q != nullptr && K != nullptr && weight != nullptr, "odit_linear_stem: null arguments");
  if (lin_engine_of(flags) != 0 || (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) != 0) return ODIT_ENOTSUP;
  GemmCall g[2];
  for (int i = 0; i < 2; ++i) {
    const LinCall c{q[i].x, q[i].w, q[i].bias, nullptr, nullptr, q[i].out, q[i].M, N, K[i], q[i].ldx, q[i].ldw, q[i].ldo, 0,
                    q[i].bias != nullptr ? ODIT_EPI_BIAS : ODIT_EPI_NONE, dtype, dtype, nullptr, 0, static_cast<hipStream_t>(stream)};
    const int rc = lin_check(c);
    if (rc != ODIT_OK) return rc;
    g[i] = lin_gemm_call(c, 0, 0);
    if (!gemm_streamk_takes(g[i], dtype) || K[i] > kSmallNormK) return ODIT_ENOTSUP;
  }
  const int most = K[0] > K[1] ? 0 : 1;  // (as many workgroups to a CU as the longer reduction's LDS leaves room for)
  GemmCall both[2] = {g[most], g[1 - most]};
  if ((K[1] & (K[1] - 1)) != 0 || !aligned16(weight) || (g[0].bias == nullptr) != (g[1].bias == nullptr) || !gemm_small_rule(both, 2, device_cus(), kSmallNormK))
    return ODIT_ENOTSUP;
  return launch_gemm_small_stem(g, weight, eps, dtype, static_cast<hipStream_t>(stream));
}

// One projection of rows that lie in two tensors, in one reduction or as two products that add up, by expected time. One
// reduction rounds once, and reads and writes the output once (M=1536, N=3072, K=12288 and 3072: 128 us, two calls 166).
extern "C" int odit_linear_join(const void* x, const void* x2, const void* w, const void* bias, void* out, const void* residual, const void* gate,
                                int M, int N, int K, int K2, int64_t ldx, int64_t ldx2, int64_t ldw, int64_t ldo, int64_t ldr, int epilogue,
                                int gate_dtype, int dtype, int rows_per_gate, int64_t gate_stride, unsigned flags, void* workspace,
                                size_t workspace_bytes, void* stream) {
  using namespace odit;
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  const LinCall c{x, w, bias, residual, gate, out, M, N, K, ldx, ldw, ldo, ldr, epilogue, gate_dtype, dtype, lib, lib_bytes, static_cast<hipStream_t>(stream)};
  const int rc = lin_check(c);
  if (rc != ODIT_OK) return rc;
  ODIT_CHECK_ARG(x2 != nullptr && K2 > 0 && ldx2 >= K2 && ldw >= K + K2, "odit_linear_join: bad second operand");
  ODIT_CHECK_ARG(rows_per_gate >= 0 && gate_stride >= 0, "odit_linear_join: rows_per_gate and gate_stride must not be negative");
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { set_error("odit_linear_join: hipGetDevice failed"); return ODIT_ELAUNCH; }
  const bool rows = lin_is_residual(c) && gate != nullptr && rows_per_gate > 0 && rows_per_gate < M;
  LinCall first = c, second = c, whole = c;  // in two calls the second one's product comes first and has the bias with it
  first.bias = nullptr;
  second.K = K2;
  second.ldx = ldx2;
  whole.K = K + K2;
  whole.clip = lin_clips(c, flags, ODIT_LINEAR_CLIP);
  const GemmCall g1 = lin_gemm_call(first, rows ? rows_per_gate : 0, rows ? gate_stride : 0), g2 = lin_gemm_call(second, g1.rows_per_gate, g1.ldg);
  GemmCall g = lin_gemm_call(whole, g1.rows_per_gate, g1.ldg);
  if (lin_engine_of(flags) != 0 || (flags & (ODIT_LINEAR_FIRST | ODIT_LINEAR_NO_TILE)) != 0 || M < kTileMinAuto || K % 64 != 0 || K2 % 64 != 0 ||
      ldx2 % 8 != 0 || !aligned16(x2) || !gemm_tile_takes(g1, dtype) || !gemm_tile_takes(g2, dtype) || !gemm_tile_takes(g, dtype))
    return ODIT_ENOTSUP;
  const TilePlan plan = plan_gemm_tile(&g, 1, device_cus(), sk != nullptr);
  if (plan.bm == 0 || plan.us >= kOneLaunchGain * (lin_call_us(dev, first, g1, sk) + lin_call_us(dev, second, g2, sk))) return ODIT_ENOTSUP;
  const TileX2 other{x2, ldx2, K};
  return launch_gemm_tile(&g, 1, &other, dtype, sk, c.stream);
}

extern "C" int odit_linear_rows_plan(const void* x, const void* w, const void* bias, void* out, const void* residual,
                                     const void* gate, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                     int64_t ldr, int epilogue, int gate_dtype, int dtype, int rows_per_gate,
                                     int64_t gate_stride, unsigned flags, void* workspace, size_t workspace_bytes,
                                     int* handwritten, int* launches) {
  using namespace odit;
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  LinCall c{x, w, bias, residual, gate, out, M, N, K, ldx, ldw, ldo, ldr, epilogue, gate_dtype, dtype,
            lib, lib_bytes, nullptr};
  int rc = lin_check(c);
  if (rc != ODIT_OK) return rc;
  ODIT_CHECK_ARG(handwritten != nullptr && launches != nullptr, "odit_linear_rows_plan: null result pointers");
  const bool per_rows = lin_is_residual(c) && gate != nullptr && rows_per_gate > 0 && rows_per_gate < M;
  const int engine = lin_engine_of(flags);
  const GemmCall g = lin_gemm_call(c, per_rows ? rows_per_gate : 0, per_rows ? gate_stride : 0);
  int dev = 0;
  (void)hipGetDevice(&dev);
  c.first = (flags & ODIT_LINEAR_FIRST) != 0;
  c.no_tile = c.first || (flags & ODIT_LINEAR_NO_TILE) != 0;
  const int kind = M == 0 || engine == 1 ? 0 : engine == 2 ? lin_handwritten_kind(g, dtype, sk) : lin_auto_kind(dev, c, g, sk);
  const bool own = kind != 0, grouped = per_rows && (!own || (kind == 4 && lin_workers(c, g) > 0));
  *handwritten = own ? 1 : 0;
  *launches = M == 0 ? 0 : (!grouped ? 1 : (M + rows_per_gate - 1) / rows_per_gate);
  if (!own && lin_needs_prep(c)) *launches *= 2;  // plus the [N]-sized gate-vector launch of the library form
  return ODIT_OK;
}

extern "C" int odit_linear(const void* x, const void* w, const void* bias, void* out, const void* residual,
                           const void* gate, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                           int64_t ldr, int epilogue, int gate_dtype, int dtype, void* workspace,
                           size_t workspace_bytes, void* stream) {
  return odit_linear_rows(x, w, bias, out, residual, gate, M, N, K, ldx, ldw, ldo, ldr, epilogue, gate_dtype, dtype, 0,
                          0, 0u, workspace, workspace_bytes, stream);
}

// Time of one launch as a tuning call compares it. A projection of a large model starts from cold caches: a flush (where a buffer is
// given) before every launch. One with a few MB of weights (kSmallWeights) belongs to a small model, whose weights stay in the
// last-level cache and whose time is often the host's: launches one after the other, as they come there (M=256, N=1024, K=1024, the
// library / the small kernel: 11.5 us / 7.6 in a row, where a library call occupies the host for longer than the GPU; 9.0 / 12.0
// behind a flush).
template <typename Launch>
static int lin_time(Launch&& launch, const odit::LinCall& c, int reps, void* flush, size_t flush_bytes, float* us) {
  const bool row = static_cast<int64_t>(c.N) * c.K < kSmallWeights;
  const int times = row ? 1 : reps, each = row ? 8 * reps : 1;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    odit::set_error("odit_linear_tune: hipEventCreate failed");
    return ODIT_ELAUNCH;
  }
  int rc = launch();
  float total = 0.f;
  for (int i = 0; i < times && rc == ODIT_OK; ++i) {
    if (!row && flush != nullptr && flush_bytes > 0) (void)hipMemsetAsync(flush, i & 0xff, flush_bytes, c.stream);
    if (row) (void)hipStreamSynchronize(c.stream);
    (void)hipEventRecord(e0, c.stream);
    for (int j = 0; j < each && rc == ODIT_OK; ++j) rc = launch();
    (void)hipEventRecord(e1, c.stream);
    if (hipEventSynchronize(e1) != hipSuccess) { odit::set_error("odit_linear_tune: hipEventSynchronize failed"); rc = ODIT_ELAUNCH; }
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    total += ms;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *us = total * 1e3f / (times * each);
  return rc;
}

// Times the library's kernels for problem c (cold caches before every timed launch when a flush buffer
// is given: in a model every projection has its own weights, which are never cache-resident, so
// back-to-back launches on one weight would rank the kernels wrongly) and keeps the fastest in the plan.
static int lin_tune_library(const odit::LinCall& c, int iters, void* flush, size_t flush_bytes, float* best_us) {
  using namespace odit;
  hipblasLtHandle_t h;
  LinPlan* p;
  const void *alpha, *cptr;
  void* lws;
  size_t lws_bytes;
  int rc = lin_prepare(c, &h, &p, &alpha, &cptr, &lws, &lws_bytes);
  if (rc != ODIT_OK) return rc;
  const hipDataType t = lin_type(c.dtype);
  std::vector<hipblasLtMatmulHeuristicResult_t> all;
  ODIT_LT(hipblaslt_ext::getAllAlgos(h, hipblaslt_ext::GemmType::HIPBLASLT_GEMM, HIPBLAS_OP_T, HIPBLAS_OP_N, t, t, t, t,
                                     HIPBLAS_COMPUTE_32F, all));
  const float beta = lin_is_residual(c) ? 1.f : 0.f;
  float best = 1e30f;
  int n_ok = 0;
  auto time_algo = [&](hipblasLtMatmulAlgo_t& algo, int reps) -> float {
    float us = 0.f;
    auto launch = [&]() -> int {
      return hipblasLtMatmul(h, p->desc, alpha, c.w, p->a, c.x, p->b, &beta, cptr, p->c, c.out, p->d, &algo, lws, lws_bytes, c.stream) ==
                     HIPBLAS_STATUS_SUCCESS ? ODIT_OK : ODIT_ELAUNCH;
    };
    return lin_time(launch, c, reps, flush, flush_bytes, &us) == ODIT_OK ? us : -1.f;
  };
  // first pass: one timed launch of every kernel the library has for these types that accepts the
  // problem; second pass: the best few again with `iters` launches each
  std::vector<std::pair<float, size_t>> ranked;
  for (size_t i = 0; i < all.size(); ++i) {
    size_t need = 0;
    if (hipblaslt_ext::matmulIsAlgoSupported(h, p->desc, alpha, p->a, p->b, &beta, p->c, p->d, all[i].algo, need) !=
            HIPBLAS_STATUS_SUCCESS || need > lws_bytes || !lin_sound(h, all[i].algo))
      continue;
    all[i].workspaceSize = need;
    const float us = time_algo(all[i].algo, 2);
    if (us > 0.f) { ranked.emplace_back(us, i); ++n_ok; }
  }
  std::sort(ranked.begin(), ranked.end());
  const size_t finalists = std::min<size_t>(ranked.size(), 12);
  for (size_t r = 0; r < finalists; ++r) {
    auto& cand = all[ranked[r].second];
    const float us = time_algo(cand.algo, iters);
    if (us > 0.f && us < best) {
      best = us;
      p->algo = cand.algo;
      p->algo_ws = cand.workspaceSize;
      p->have_algo = true;
      p->tuned = true;
    }
  }
  if (n_ok == 0) {
    set_error("odit_linear_tune: none of the library's %zu kernels accepts this problem", all.size());
    return ODIT_ENOTSUP;
  }
  *best_us = best;
  return ODIT_OK;
}

extern "C" int odit_linear_rows_tune(const void* x, const void* w, const void* bias, void* out, const void* residual,
                                     const void* gate, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                     int64_t ldr, int epilogue, int gate_dtype, int dtype, int rows_per_gate,
                                     int64_t gate_stride, void* workspace, size_t workspace_bytes, void* stream,
                                     int iters, void* flush, size_t flush_bytes, float* best_us, int* handwritten) {
  using namespace odit;
  if (handwritten) *handwritten = 0;
  void *sk, *lib;
  size_t lib_bytes;
  lin_split_ws(workspace, workspace_bytes, &sk, &lib, &lib_bytes);
  LinCall c{x, w, bias, residual, gate, out, M, N, K, ldx, ldw, ldo, ldr, epilogue, gate_dtype, dtype,
            lib, lib_bytes, static_cast<hipStream_t>(stream)};
  int rc = lin_check(c);
  if (rc != ODIT_OK) return rc;
  ODIT_CHECK_ARG(M > 0 && iters > 0, "odit_linear_tune: needs M > 0 and iters > 0");
  ODIT_CHECK_ARG(rows_per_gate >= 0 && gate_stride >= 0, "odit_linear_tune: rows_per_gate and gate_stride must not be negative");
  const bool per_rows = lin_is_residual(c) && gate != nullptr && rows_per_gate > 0 && rows_per_gate < M;
  const GemmCall g = lin_gemm_call(c, per_rows ? rows_per_gate : 0, per_rows ? gate_stride : 0);
  const int rule = lin_rule_kind(c, g, sk);  // (before the library's plans hold what is tuned)
  // the library runs one launch per group of rows: tune that launch (on the first group), and the shorter
  // launch of a last group that is not full, which is a problem of its own to the library
  LinCall cl = c;
  int launches = 1, last_rows = 0;
  if (per_rows) {
    cl.M = rows_per_gate;
    launches = M / rows_per_gate;
    last_rows = M % rows_per_gate;
  }
  float lib_us = 0.f;
  rc = lin_tune_library(cl, iters, flush, flush_bytes, &lib_us);
  if (rc != ODIT_OK) return rc;
  lib_us *= static_cast<float>(launches);
  if (last_rows > 0) {
    LinCall cr = cl;   // (timed on the first rows: only the shape matters)
    cr.M = last_rows;
    float last_us = 0.f;
    rc = lin_tune_library(cr, iters, flush, flush_bytes, &last_us);
    if (rc != ODIT_OK) return rc;
    lib_us += last_us;
  }
  // two kernels' times less than 3 % apart say nothing about their times in a model: the rule's choice stays
  constexpr float kSame = .97f;
  Tuned best{0, lib_us};
  float best_at = rule == 0 ? kSame * lib_us : lib_us;
  bool compared = false;
  for (int kind = 1; kind <= 3; ++kind) {
    if (!lin_candidate(kind, g, dtype, sk)) continue;
    float own_us = 0.f;
    rc = lin_time([&]() -> int { return lin_launch_handwritten(kind, g, dtype, sk, c.stream); }, c, iters, flush, flush_bytes, &own_us);
    if (rc != ODIT_OK) return rc;
    compared = true;
    const float at = kind == rule ? kSame * own_us : own_us;
    if (at < best_at) {
      best = Tuned{kind, own_us};
      best_at = at;
    }
  }
  if (compared) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lock(g_engine_mu);
    g_tuned[lin_tuned_key(dev, c, g.rows_per_gate, sk)] = best;
  }
  if (handwritten) *handwritten = best.kind != 0 ? 1 : 0;
  if (best_us) *best_us = best.us;
  return ODIT_OK;
}

extern "C" int odit_linear_tune(const void* x, const void* w, const void* bias, void* out, const void* residual,
                                const void* gate, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                int64_t ldr, int epilogue, int gate_dtype, int dtype, void* workspace,
                                size_t workspace_bytes, void* stream, int iters, void* flush,
                                size_t flush_bytes, float* best_us) {
  return odit_linear_rows_tune(x, w, bias, out, residual, gate, M, N, K, ldx, ldw, ldo, ldr, epilogue, gate_dtype, dtype,
                               0, 0, workspace, workspace_bytes, stream, iters, flush, flush_bytes, best_us, nullptr);
}
