// 16-bit GEMM y = x W^T for projections with many rows, for one problem or up to three of the same reduction length in one launch.
//
// Workgroup: 8 wavefronts, two per SIMD, on an output tile of BM x BN = 256 x 256 (or 128 x 256). The tile's rows are two
// halves X0, X1 and its features two halves W0, W1; a wavefront (2 along the rows x 4 along the features) owns a quarter of
// each of the four quadrants, as v_mfma_f32_16x16x32 accumulators with W rows as the A operand.
//
// Anti-phase. Wavefronts w and w + 4 share a SIMD. A reduction step of 64 is two phases, rows X0 and rows X1, and each phase
// is a slot of LDS reads and tile loads followed by a slot of 32 matrix instructions. A barrier ends every slot and the second
// four wavefronts run one slot behind the first four, so on every SIMD one wavefront multiplies while the other one reads: the
// fragment reads (192 KB per step through an LDS that moves 128 bytes per cycle: 1536 cycles) and the tile loads (64 KB)
// proceed beside the 2048 cycles of matrix work. The predecessor of this kernel ran its 8 wavefronts in one phase and took
// one after the other: 1.08 to 1.14 PFLOP/s.
//
// Tile movement. A step is four units X0, X1, W0, W1 of 128 rows x 128 bytes, moved from global memory straight into LDS by
// `buffer_load_dwordx4 ... lds` (one wave instruction fills 1 KB = 8 rows; the lane chooses WHAT it fetches, a 16-byte chunk
// whose number is XORed with bits of the row, so that the 16-byte fragment reads of 16 rows cover all 64 banks). A unit is
// read in one phase only and both groups of wavefronts have waited for their reads when that phase's slots end, so it is
// refilled from the next phase on, with the data of two steps later: every load has three phases (about 3000 cycles) to
// arrive, and a wavefront never waits for its last loads. The loads go out one by one between the fragment reads: in one
// burst they queue up in front of the texture addresser (16 cycles per instruction) and hold the reads behind them up (N=8192,
// K=8192, M=8192: 1.48 PFLOP/s in one burst, 1.55 between the reads; among the matrix instructions 1.43: they come too late).
//
// The workgroup is persistent and the stream of steps does not stop at a tile's end: the next tile's first units are on their
// way while this tile's epilogue runs. Tiles are dealt out round by round. The tiles of a last round that would leave half or
// more of the compute units without work are cut along the reduction instead, into 2 to 4 equal parts (of tiles of 128 rows up to 8), behind the whole tiles.
// The parts of a tile share its four quadrants out between them (from the fifth on they have none): each leaves its fp32 sums for the others' quadrants
// in scratch (write-through), keeps its own ones' in LDS and takes a ticket; when all have arrived it adds up all sums of its quadrants,
// in the order of the parts (the result does not depend on who arrives when), and runs their epilogue. A part that does not find
// the others arrived after a bounded number of looks leaves its own sums in scratch too and goes, and the last to arrive takes
// what is left: nobody waits for anybody without a bound. Ticket words carry the launch's epoch (see gemm_bf16.hip). What the
// parts cost is the traffic of their sums (2 x 256 KB for each of them if all go through memory). us, one workgroup adding all up /
// each its quadrants, all through memory and parts ahead of the whole tiles / as described: M=512, N=3072, K=12288 in 4 parts
// 77 / 60 / 55; M=512, N=9216, K=3072 in 3 - / 48.5 / 41.5; M=8192, N=9216, K=3072, half a round in 2 parts - / 338 / 323. (With the
// parts of a tile on one XCD and its L2 in the place of memory: the same time or 2 us more.)
//
// Epilogue: W rows are assigned to accumulators so that a lane ends up with 8 consecutive features of one output row, stored
// as 16 bytes from registers; bias, GELU(tanh), gate and residual are applied on the way.
//
// What bounds it: the matrix pipe and the clock that the part holds under it. 8192 x 8192 x 8192 on random operands takes 1.35
// us per step of 256 x 256 x 64 (1.59 PFLOP/s; hipBLASLt 1.60 on that card), 1.23 where one round runs. Measured with cold
// weights, us, this kernel / its predecessor (256 x 256 or 256 x 192 tiles, 8 wavefronts in one phase) / the library's choice:
// M=8192, N=12288, K=3072 with GELU 440 / 543 / 447; M=8192, N=9216, K=3072 323 / 402 / 437; M=2706, N=5120, K=5120 107 / 135 /
// 117; M=2706, N=13824, K=5120 with GELU 289 / 399 / 319; M=1536, N=9216, K=3072 68 / 89 / 72. Around the loop a launch costs 3 us,
// a tile's end 6 (9 with GELU: its arithmetic has no matrix work to hide behind).
#pragma once

#include <algorithm>
#include <type_traits>

#include "gemm_epilogue.h"
#include "gemm_heads.h"

namespace odit {

namespace {

constexpr int kTileN = 256;                      // features per tile
constexpr int kTileK = 64;                       // reduction elements per step
constexpr int kTileSlot = 256 * kTileN * 4;      // bytes of a partial tile
static_assert(static_cast<size_t>(kTileSlot) * kGemmMaxWorkers + kGemmCounterBytes <= kGemmScratchBytes, "one slot per workgroup");

struct TileProblem {
  const void *x, *w;
  // reduction steps from `k_split` on take their x from x2
  const void* x2;
  int M, N, k_split;
  uint32_t ldx, ldx2, ldw;  // bytes
  uint32_t x_bytes, x2_bytes, w_bytes;
  int m_tiles, n_tiles;
  int x_last, w_last;  // rows to fetch a tile's past rows from at most (fill_tile_params)
  GemmEpilogue ep;
};

struct TileParams {
  TileProblem q[3];
  int tiles0, tiles1, tiles;  // tiles of the first problem, of the first two, of all
  int whole;          // tiles that are not cut; the others are cut into `parts` along the reduction
  int parts;
  int k_steps;
  unsigned long long* counters;  // one ticket word per cut tile, zero between launches
  unsigned long long epoch;      // larger than that of any earlier launch of the process
  char* slots;
};

template <bool HEADS, bool UNLESS, bool SHARED = false> struct TileArgs : TileParams {};
template <> struct TileArgs<true, false> : TileParams {
  HeadsOut heads[2];  // of the two problems (there are no three with heads); q null: an ordinary output
};
template <> struct TileArgs<false, true> : TileParams {
  const int* unless;
};
// The steps of the tiles from `shared` on are shared out one tile after the other, `share` steps to a worker and one more to the first `more` of them. A tile
// that several of them have a share of is the sum of their sums, in their order. (share 0: all tiles are whole, and shared == tiles)
template <> struct TileArgs<false, false, true> : TileParams {
  int shared, share, more;
};

typedef __attribute__((address_space(3))) void* lds_void_p;

// A wave-uniform number in a scalar register, where the compiler would not keep it by itself.
__device__ __forceinline__ int scalar(int a) {
  int s = __builtin_amdgcn_readfirstlane(a);
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+s"(s));
#endif
  return s;
}
// a / b of wave-uniform numbers (the division runs on the vector unit, and what follows from its result would stay there, buffer
// descriptors included)
__device__ __forceinline__ int quotient(int a, int b) { return scalar(static_cast<int>(static_cast<unsigned>(a) / static_cast<unsigned>(b))); }

constexpr int kThrough = 16;  // sc1 of a buffer access: past the XCD's L2, as an agent-scope store or load of a word goes
// Ticket word of a cut tile: arrivals in bits 0 to 3, quadrants given up 4 to 7, departures 8 to 11, the launch's epoch from 16 on
constexpr unsigned long long kArrival = 1, kDeparture = 1 << 8;
constexpr int kLooks = 64;    // looks for the other parts of a tile, about a microsecond each
// Parts of a tile of 128 rows and of 256 at most. Beyond four (the sums of 8 parts of a quadrant fit the registers of the lower tiles only), cold weights,
// us, stream-K / 4 parts / this many: N=3072, K=12288: M=256 47.1 / 54.8 / 8: 41.3, 300 47.3 / 49.3 / 7: 43.2, 512 55.6 / 56.6 / 5: 52.7, 195 + 256
// 62.2 / 63.1 / 5: 58.7, 128 + 40 51.5 / 59.4 / 8: 46.5; K=15360: 300 56.4 / 60.0 / 7: 48.8, 451 69.3 / 62.8 / 5: 58.9; N=5120, K=13824: 256
// 67.0 / 63.5 / 6: 53.9. Short reductions gain nothing: N=3072, K=3072: 256 + 64 22.8 / 24.8 / 5: 24.4.
constexpr int kMaxParts[2] = {8, 4};

// What the epilogue of a problem is to a tile with rows m0 .. m0 + BM - 1: 0 bias, 1 bias and GELU, 2 gate and residual, 3 the
// same where gate vectors change inside the tile
__device__ __forceinline__ int epilogue_kind(const GemmEpilogue& e, int m0, int bm) {
  if (e.epilogue == ODIT_EPI_GATED_RESIDUAL || e.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE) {
    const int last = m0 + bm < e.M ? m0 + bm - 1 : e.M - 1;
    return e.rows_per_gate > 0 && quotient(m0, e.rows_per_gate) != quotient(last, e.rows_per_gate) ? 3 : 2;
  }
  return e.epilogue == ODIT_EPI_GELU_TANH || e.epilogue == ODIT_EPI_BIAS_GELU_TANH ? 1 : 0;
}

// All loads have arrived, on every path: without it the compiler, which sees paths around the use of a loaded value, waits for
// it where the register is written next, inside the main loop, and there for the tile loads in flight too (+25 % on a step).
__device__ __forceinline__ void loads_arrived() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)

// A gated or residual result (APART: in the library's order of operations)
template <typename T, bool APART>
__device__ __forceinline__ float gated_result(const GemmEpilogue& e, float a, float gate, float bias, float residual) {
  return gemm_clipped<T>(e, APART ? gemm_gated_apart(a, gate, residual, bias) : fmaf(gate, a, bias) + residual);
}

// This lane's part of a quadrant of a tile: 8 features from n on of the rows m, m + 16, ...
template <typename T, int MH, int K, bool APART>
__device__ __forceinline__ void finish_quadrant(const GemmEpilogue& e, int m0, int m, int n, const f32x4_v (&v)[MH][2]) {
  const bool in = n < e.N;
  if constexpr (K == 3) {
    // Two rows a round trip to memory, each with its gate vector. (Row by row a quadrant is four trips one after the other, and where a launch
    // is one round its end waits for such a tile: 2048 + 342 rows, two gate vectors each, N=3072, K=3072 59.9 us, now 56.6. More rows at
    // once do not fit beside the sums.)
#pragma unroll
    for (int i0 = 0; i0 < MH; i0 += 2) {
      float gt[2][8], bs[2][8];
      u32x4 res[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = m + (i0 + j) * 16 < e.M ? m + (i0 + j) * 16 : e.M - 1;
        gemm_epilogue_vectors8<T>(e, row, in ? n : 0, gt[j], bs[j]);
        res[j] = load_raw(static_cast<const T*>(e.residual) + row * e.ldr + (in ? n : 0));
      }
      loads_arrived();
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        u32x4 o;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const f32x4_v a = v[i0 + j][u >> 1];
          Raw<T>::set2(o, u, gated_result<T, APART>(e, a[2 * (u & 1)], gt[j][2 * u], bs[j][2 * u], Raw<T>::get(res[j], 2 * u)),
                       gated_result<T, APART>(e, a[2 * (u & 1) + 1], gt[j][2 * u + 1], bs[j][2 * u + 1], Raw<T>::get(res[j], 2 * u + 1)));
        }
        if (in && m + (i0 + j) * 16 < e.M) store_raw(static_cast<T*>(e.out) + (m + (i0 + j) * 16) * e.ldo + n, o);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    float gt[8], bs[8];
    gemm_epilogue_vectors8<T>(e, m0, in ? n : 0, gt, bs);
    u32x4 res[MH];
    if constexpr (K == 2) {
#pragma unroll
      for (int i = 0; i < MH; ++i) {
        const int row = m + i * 16 < e.M ? m + i * 16 : e.M - 1;
        res[i] = load_raw(static_cast<const T*>(e.residual) + row * e.ldr + (in ? n : 0));
      }
    }
    loads_arrived();
#pragma unroll
    for (int i = 0; i < MH; ++i) {
      float y[8];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        y[u] = v[i][0][u];
        y[4 + u] = v[i][1][u];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if constexpr (K == 2) y[u] = gated_result<T, APART>(e, y[u], gt[u], bs[u], Raw<T>::get(res[i], u));
        else y[u] += bs[u];
        if constexpr (K == 1) y[u] = APART ? gemm_gelu_apart(y[u]) : gemm_gelu_tanh(y[u]);
      }
      u32x4 o;
#pragma unroll
      for (int u = 0; u < 4; ++u) Raw<T>::set2(o, u, y[2 * u], y[2 * u + 1]);
      if (in && m + i * 16 < e.M) store_raw(static_cast<T*>(e.out) + (m + i * 16) * e.ldo + n, o);
    }
  }
}
template <typename T, int MH, bool UNGATED, bool APART>
__device__ __forceinline__ void finish_quadrant(int kind, const GemmEpilogue& e, int m0, int m, int n, const f32x4_v (&v)[MH][2]) {
  if (kind == 0) finish_quadrant<T, MH, 0, APART>(e, m0, m, n, v);
  else if (UNGATED || kind == 1) finish_quadrant<T, MH, 1, APART>(e, m0, m, n, v);
  else if (kind == 2) finish_quadrant<T, MH, 2, APART>(e, m0, m, n, v);
  else finish_quadrant<T, MH, 3, APART>(e, m0, m, n, v);
}

// ---- query, key and value heads (HeadsOut): the end of a quadrant in two passes with a barrier between them ----
// The projection's values as they would be stored, which take the registers of the sums, and what this wavefront's 32 features add to
// the squares of their head's row: squares[row][wavefront along the features]. r: the lane's first row in the tile. (Row by row: what
// the compiler would form of all rows at once does not fit beside the sums.)
template <typename T, int MH>
__device__ __forceinline__ void square_heads(const f32x4_v (&v)[MH][2], u32x4 bias, u32x4 (&x)[MH], float* squares, int r, int wn, int lq) {
#pragma unroll
  for (int i = 0; i < MH; ++i) {
#pragma unroll
    for (int u = 0; u < 4; ++u) Raw<T>::set2(x[i], u, v[i][u / 2][2 * (u % 2)] + Raw<T>::get(bias, 2 * u), v[i][u / 2][2 * (u % 2) + 1] + Raw<T>::get(bias, 2 * u + 1));
    asm volatile("" : "+v"(x[i]));
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) s = fmaf(Raw<T>::get(x[i], u), Raw<T>::get(x[i], u), s);
    asm volatile("" : "+v"(x[i]));  // (unpacked again in the second pass and not kept so)
    s = add_swapped(s, __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false));
    s = add_swapped(s, __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false));
    squares[(r + i * 16) * 4 + wn] = s;  // (the same from four lanes: a branch here costs the registers of all sums behind it)
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The second pass, features f .. f + 7: norm over the head, weight, rotation (queries and keys), and the store. The sums of squares are
// added in the order of qknorm_flat_kernel.
template <typename T, int MH>
__device__ __forceinline__ void store_heads(const HeadsOut& h, const u32x4 (&v)[MH], const HeadRows<MH>& rows, const float* squares, int r, int wn, int third,
                                            int f, u32x4 weight) {
  T* const out = static_cast<T*>(third == 0 ? h.q : third == 1 ? h.k : h.v) + (f - third * h.HD);
#pragma unroll
  for (int i = 0; i < MH; ++i) {
    u32x4 o = v[i];
    if (third < 2) {
      const f32x4_v s = *reinterpret_cast<const f32x4_v*>(squares + (r + i * 16) * 4);
      const float lo = s[0] + s[1], hi = s[2] + s[3];
      const float sum = h.D == 128 ? lo + hi : (wn & 2 ? hi : lo);
      const float rstd = rsqrtf(sum * (h.D == 128 ? 1.f / 128 : 1.f / 64) + h.eps);
      o = turn_head<T>(v[i], rstd, weight, rows.cos[i], rows.sin[i]);
    }
    if (rows.at[i] >= 0) store_raw(out + static_cast<int64_t>(rows.at[i]) * h.HD, o);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// MH: 16-row accumulators of a wavefront in each half of the rows (4: 256-row tiles, 2: 128). HEADS: the form for problems whose
// output is query, key and value heads, beside ordinary ones without a gate. UNLESS: nothing is done where a word of device memory is not 0 (a
// form of its own, as the test made the others up to 0.6 % slower: M=1536, N=12288, K=3072 109.7 / 110.4 us). APART: gemm_gated_apart and gemm_gelu_apart (likewise), and
// no tile in parts. SHARED: TileArgs's shared tiles, each by one workgroup.
template <typename T, int MH, bool HEADS, bool UNLESS, bool APART = false, bool SHARED = false>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tile_kernel(const TileArgs<HEADS, UNLESS, SHARED> p) {
  using M = Mma16<T>;
  using frag = typename M::frag;
  constexpr int BM = 64 * MH, HM = 32 * MH;           // rows of a tile, of a half
  constexpr int kXUnit = HM * 128, kWUnit = 128 * 128;
  constexpr int kStage = 2 * (kXUnit + kWUnit);
  constexpr int XJ = MH / 2, WJ = 2, PJ = XJ + WJ;    // tile-load instructions of a wavefront per unit, per phase
  constexpr int NR = 2 * MH + 4;                      // fragment reads per phase
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStage + 64 + (HEADS ? 2 * BM * 16 : 0)];
  int* const flag = reinterpret_cast<int*>(lds + 2 * kStage);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;  // (wm is also the group: the second four wavefronts run a slot behind)
  const int l16 = lane & 15, lq = lane >> 4;
  const int G = gridDim.x;
  const int v = xcd_remap(blockIdx.x, G);
  const int nk = p.k_steps;
  if constexpr (UNLESS) {
    if (*p.unless != 0) return;  // (the whole launch: no ticket is drawn)
  }

  auto make_rsrc = [](const void* base, uint32_t bytes) __attribute__((always_inline)) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    u32x4_v r;
    r.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    r.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32) & 0xffffu);
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;
    return r;
  };

  // problem, first row and first feature of a tile: groups of 8 row tiles, feature tiles outer inside a group, so that the 32
  // tiles an XCD runs at a time share 8 pieces of x and 4 of W (SHARED: of 16, the order in which they are shared out, which costs 1 to 4 % of a
  // large launch: all tiles whole, us, groups of 8 / 16: 65520 rows, N=13824, K=5120 with GELU 6136 / 6395, N=15360 6779 / 6939; 7072 rows, N=15360 777 / 790)
  constexpr int kGroup = SHARED ? 16 : 8;
  auto locate = [&](int tile, int& which, int& m0, int& n0) __attribute__((always_inline)) {
    which = tile >= p.tiles1 ? 2 : tile >= p.tiles0 ? 1 : 0;
    const int t = tile - (which == 2 ? p.tiles1 : which == 1 ? p.tiles0 : 0);
    const int mt = p.q[which].m_tiles, per = kGroup * p.q[which].n_tiles;
    const int g = quotient(t, per), first = g * kGroup, gm = mt - first < kGroup ? mt - first : kGroup;
    const int r = t - g * per, nt = quotient(r, gm);
    m0 = (first + r - nt * gm) * BM;
    n0 = nt * kTileN;
  };
  // The segments of this workgroup: whole tiles, then its part of a cut tile. A cursor is (part still to do, next whole tile).
  const int cut = p.tiles - p.whole;
  const bool has_part = !APART && v < cut * p.parts;
  // quadrants that this part of a cut tile finishes: its number's, and the one `parts` further
  auto quadrants = [&]() __attribute__((always_inline)) -> int {
    const int part = quotient(v, cut);
    return scalar((part < 4 ? 1 << part : 0) | (part + p.parts < 4 ? 1 << (part + p.parts) : 0));
  };
  constexpr int kQuad = 2 * MH * 8192;  // bytes of a quadrant's accumulators
  // SHARED: no tile is cut; the next tile's steps from `at` on are to come, each worker's a segment.
  struct Cursor { bool part; int next, at = 0; };
  auto next_segment = [&](Cursor& c, int& tile, int& k0, int& k1) __attribute__((always_inline)) -> bool {
    if constexpr (SHARED) {
      if (c.next >= p.tiles) return false;
      tile = c.next;
      k0 = c.at;
      k1 = nk;
      if (tile >= p.shared) {
        const int from = (tile - p.shared) * nk + k0, longer = p.more * (p.share + 1);
        const int to = from < longer ? (quotient(from, p.share + 1) + 1) * (p.share + 1) : longer + (quotient(from - longer, p.share) + 1) * p.share;
        if (to - from < nk - k0) k1 = scalar(k0 + to - from);
      }
      c.at = k1 < nk ? k1 : 0;
      if (c.at == 0) c.next += G;
      return true;
    }
    if (c.next < p.whole) {
      tile = c.next;
      c.next += G;
      k0 = 0;
      k1 = nk;
      return true;
    }
    if (!c.part) return false;
    c.part = false;
    const int part = quotient(v, cut);
    tile = p.whole + v - part * cut;
    k0 = quotient(part * nk, p.parts);
    k1 = quotient((part + 1) * nk, p.parts);
    return true;
  };

  // ---- tile loads ----
  // Instruction j of this wavefront's share of a unit fills rows (wave * J + j) * 8 .. + 7; lane l lands in row + l / 8, chunk
  // l % 8, and fetches chunk (l % 8) ^ swizzle(row). The products of rows past the end (fill_tile_params) land in output rows
  // and features that are never stored.
  // (the lane's number is hidden from the compiler wherever a segment begins or ends: it would form what follows from it once in
  // front of everything and keep it in registers that the main loop needs)
  auto hidden_lane = [&]() __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  u32x4_v xr, wr;
  uint32_t vx[2][XJ], vw[2][WJ];  // byte offsets of the lane's chunks (X0, X1; W0, W1)
  constexpr int advance = kTileK * 2;
  int kx = 0, kw = 0;             // byte offset of the step along x and W rows
  int left = 0, rest = 0, pq = 0, pm0 = 0;  // steps until x changes its source or the segment ends; behind that
  Cursor pc{has_part, v};
  auto x_rows = [&](const void* x, uint32_t bytes, uint32_t ld, int last) __attribute__((always_inline)) {
    xr = make_rsrc(x, bytes);
    const int ln = hidden_lane(), lrow = ln >> 3, lch = ln & 7;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < XJ; ++j) {
        const int r = (wave * XJ + j) * 8 + lrow;
        int row = pm0 + h * HM + r;
        row = row < last ? row : last;
        vx[h][j] = static_cast<uint32_t>(row) * ld + static_cast<uint32_t>((lch ^ ((r >> 1) & 7)) << 4);
      }
  };
  auto fetch_from = [&]() __attribute__((always_inline)) {  // the next segment, or nowhere
    int tile = 0, k0 = 0, k1 = 1 << 29, n0;
    // (behind the last segment two more steps are fetched, which nobody uses: from the first row of x and of W, a few steps
    // into which are in range whatever the row's length, as there are 8 rows or more)
    const bool any = next_segment(pc, tile, k0, k1);
    locate(tile, pq, pm0, n0);
    const TileProblem& q = p.q[pq];
    wr = make_rsrc(q.w, q.w_bytes);
    const int ln = hidden_lane(), lrow = ln >> 3, lch = ln & 7;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const int r = (wave * WJ + j) * 8 + lrow, last = any ? q.w_last : 0;
        int row = n0 + h * 128 + r;
        row = row < last ? row : last;
        vw[h][j] = static_cast<uint32_t>(row) * q.ldw + static_cast<uint32_t>((lch ^ (((r >> 1) & 1) | (((r >> 3) & 3) << 1))) << 4);
      }
    pq = scalar(pq);
    pm0 = scalar(pm0);
    kw = scalar(k0 * (kTileK * 2));
    const bool far = k0 >= q.k_split;
    x_rows(far ? q.x2 : q.x, far ? q.x2_bytes : q.x_bytes, far ? q.ldx2 : q.ldx, any ? q.x_last : 0);
    kx = scalar((far ? k0 - q.k_split : k0) * (kTileK * 2));
    rest = scalar(any && !far && k1 > q.k_split ? k1 - q.k_split : 0);
    left = scalar(k1 - k0 - rest);
  };
  // the step behind the last one of the segment, or of a source of x
  auto next_source = [&]() __attribute__((always_inline)) {
    if (rest > 0) {
      const TileProblem& q = p.q[pq];
      x_rows(q.x2, q.x2_bytes, q.ldx2, q.x_last);
      kx = scalar(0);
      kw = scalar(kw + advance);
      left = scalar(rest);
      rest = scalar(0);
    } else {
      fetch_from();
    }
  };
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_p)lds));
  auto load = [&](uint32_t dst, uint32_t off, u32x4_v rs, int soff) __attribute__((always_inline)) {
    load_lds16(__builtin_amdgcn_readfirstlane(dst), off, rs, scalar(soff));
  };
  auto load_x = [&](int stage, int h, int j) __attribute__((always_inline)) { load(lds0 + stage * kStage + h * kXUnit + (wave * XJ + j) * 1024, vx[h][j], xr, kx); };
  auto load_w = [&](int stage, int h, int j) __attribute__((always_inline)) { load(lds0 + stage * kStage + 2 * kXUnit + h * kWUnit + (wave * WJ + j) * 1024, vw[h][j], wr, kw); };

  // ---- fragments ----
  // x: rows (wave's first row of the half) + 16 m + l16, chunk 4 ks + lq. W: accumulator n of a half takes the features whose
  // bit 2 is n out of the wavefront's 32, so that n = 0 and 1 together give a lane 8 consecutive ones.
  const int xrow = wm * (16 * MH) + l16;
  const int xa = xrow * 128 + ((lq ^ ((xrow >> 1) & 7)) << 4);
  const int wrow = wn * 32 + ((l16 >> 2) << 3) + (l16 & 3);
  const int wa = 2 * kXUnit + wrow * 128 + ((lq ^ (((wrow >> 1) & 1) | (((wrow >> 3) & 3) << 1))) << 4);
  f32x4_v acc[2][2][MH][2];  // half of the rows, half of the features
  frag xf[2][MH], w0[2][2], w0b[2][2], w1[2][2];
  auto read_w = [&](int stage, int h, frag (&w)[2][2], int ks, int n) {
    w[ks][n] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(lds + stage * kStage + (wa ^ (ks * 64)) + h * kWUnit + n * 512));
  };
  auto read_x = [&](int stage, int h, int ks, int m) __attribute__((always_inline)) {
    xf[ks][m] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(lds + stage * kStage + (xa ^ (ks * 64)) + h * kXUnit + m * 2048));
  };
  // A phase's reads (half h of the rows from `stage`, half wh of the features from `w_stage`) with its tile loads in between
  auto reads = [&](int stage, int h, int w_stage, int wh, frag (&w)[2][2], auto&& load_number) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int ks = r / (NR / 2), i = r % (NR / 2);
      // one W fragment, MH / 2 of x, and again
      const int g = i / (1 + MH / 2), o = i % (1 + MH / 2);
      if (o == 0) read_w(w_stage, wh, w, ks, g);
      else read_x(stage, h, ks, g * (MH / 2) + o - 1);
      if ((r + 1) * PJ / NR > r * PJ / NR) {
        __builtin_amdgcn_sched_barrier(0);
        load_number(r * PJ / NR);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // this wavefront's reads are in registers, and its loads of all but the last two phases have landed
  auto slot_wait = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * PJ) : "memory");
  };
  auto multiply = [&](int h, frag (&w0)[2][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int m = 0; m < MH; ++m)
#pragma unroll
          for (int n = 0; n < 2; ++n) acc[h][b][m][n] = M::run(b ? w1[ks][n] : w0[ks][n], xf[ks][m], acc[h][b][m][n]);
  };

  auto has_heads = [&](int which) __attribute__((always_inline)) {
    // (a scalar: were it a lane's, both sides would be run one after the other, with the sums kept through the first)
    if constexpr (HEADS) return scalar(p.heads[which].q != nullptr) != 0;
    else return false;
  };
  // a whole tile of query, key and value heads (rows in the order of the halves)
  float* const squares = reinterpret_cast<float*>(lds + 2 * kStage + 64);  // (HEADS)
  auto finish_heads = [&](const HeadsOut& hd, const GemmEpilogue& e, int m0, int n0, int ln) __attribute__((always_inline)) {
    const int r = wm * (16 * MH) + (ln & 15), q = ln >> 4, f = n0 + wn * 32 + q * 8, d = f & (hd.D - 1);
    u32x4 bias[2], weight[2];
    int third[2];
    u32x4 x[2][2][MH];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      third[b] = quotient(n0 + b * 128 + wn * 32, hd.HD);
      bias[b] = weight[b] = u32x4{0u, 0u, 0u, 0u};
      if (e.bias != nullptr && third[b] < 3) bias[b] = load_raw(static_cast<const T*>(e.bias) + f + b * 128);
      if (third[b] < 2) weight[b] = load_raw(static_cast<const T*>(third[b] == 0 ? hd.wq : hd.wk) + d);
    }
    loads_arrived();
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) square_heads<T, MH>(acc[h][b], bias[b], x[h][b], squares + b * BM * 4, r + h * HM, wn, q);
    HeadRows<MH> rows[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rows[h].ask(hd, e.M, m0, r + h * HM, d);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
    loads_arrived();
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (third[b] < 3) store_heads<T, MH>(hd, x[h][b], rows[h], squares + b * BM * 4, r + h * HM, wn, third[b], f + b * 128, weight[b]);
  };

  // step 0 and all of step 1 that its first phases do not load, in the order of the main loop
  fetch_from();
#pragma unroll
  for (int j = 0; j < WJ; ++j) load_w(0, 0, j);
#pragma unroll
  for (int j = 0; j < XJ; ++j) load_x(0, 0, j);
#pragma unroll
  for (int j = 0; j < WJ; ++j) load_w(0, 1, j);
#pragma unroll
  for (int j = 0; j < XJ; ++j) load_x(0, 1, j);
  if (left > 1) {
    left = scalar(left - 1);
    kx = scalar(kx + advance);
    kw = scalar(kw + advance);
  } else {
    next_source();
  }
#pragma unroll
  for (int j = 0; j < WJ; ++j) load_w(1, 0, j);
#pragma unroll
  for (int j = 0; j < XJ; ++j) load_x(1, 0, j);
#pragma unroll
  for (int j = 0; j < WJ; ++j) load_w(1, 1, j);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PJ) : "memory");
  barrier();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int n = 0; n < 2; ++n) read_w(0, 0, w0, ks, n);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  barrier();  // W0 of step 0 is read: the first phase refills it

  Cursor cc{has_part, v};
  int tile, k0, k1;
  bool more = next_segment(cc, tile, k0, k1);
  int st = 0;  // stage of the step
  while (more) {
    if (wm == 1) barrier();  // a slot behind
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int m = 0; m < MH; ++m)
#pragma unroll
          for (int n = 0; n < 2; ++n) acc[h][b][m][n] = f32x4_v{0.f, 0.f, 0.f, 0.f};
    // One step; `turn`: the loads leave their segment (or x its source) in the middle of it. Most steps do not, and their loop
    // holds nothing but additions beside the reads, loads and matrix instructions.
    auto step = [&](int stage, frag (&w0)[2][2], frag (&w0_next)[2][2], auto turn) __attribute__((always_inline)) {
      // rows X0 of this step; loads: X1 of the next step, W0 of the one after
      reads(stage, 0, stage, 1, w1, [&](int d) __attribute__((always_inline)) {
        if (d < XJ) {
          load_x(stage ^ 1, 1, d);
        } else {
          if (d == XJ) {
            if constexpr (decltype(turn)::value) {
              next_source();
            } else {
              kx = scalar(kx + advance);
              kw = scalar(kw + advance);
            }
          }
          load_w(stage, 0, d - XJ);
        }
      });
      slot_wait();
      barrier();
      multiply(0, w0);
      barrier();
      // rows X1 of this step and W0 of the next; loads: X0 and W1 of the one after
      reads(stage, 1, stage ^ 1, 0, w0_next, [&](int d) __attribute__((always_inline)) {
        if (d < XJ) load_x(stage, 0, d);
        else load_w(stage, 1, d - XJ);
      });
      slot_wait();
      barrier();
      multiply(1, w0);
      barrier();
    };
    auto one = [&](auto turn) __attribute__((always_inline)) {
      step(st, w0, w0b, turn);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int n = 0; n < 2; ++n) w0[ks][n] = w0b[ks][n];
      st ^= 1;
    };
    for (int todo = k1 - k0; todo > 0;) {
      int plain = scalar(todo < left - 1 ? todo : left - 1);
      todo -= plain;
      left = scalar(left - plain);
      for (; plain > 1; plain -= 2) {  // W0 in two sets of registers by turns
        step(st, w0, w0b, std::false_type{});
        step(st ^ 1, w0b, w0, std::false_type{});
      }
      if (plain > 0) one(std::false_type{});
      if (todo > 0) {
        one(std::true_type{});
        --todo;
      }
    }
    if (wm == 0) barrier();  // both groups are here

    bool whole = k0 == 0 && k1 == nk;
    if constexpr (SHARED) {
      if (!whole) {
        // The sum so far of a shared tile waits in this workgroup's slot for the next piece's, each thread's own accumulators. (no store with a scalar offset: see below)
        const auto slot = __builtin_amdgcn_make_buffer_rsrc(p.slots + static_cast<int64_t>(v) * kTileSlot, 0, kTileSlot, 0x00020000);
        const uint32_t own = static_cast<uint32_t>((wave * 64 + hidden_lane()) * 16);
        whole = k1 == nk;
#pragma unroll
        for (int quad = 0; quad < 4; ++quad) {
          if (k0 != 0) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {  // (all at once would not fit the registers)
              f32x4_v before[MH];
#pragma unroll
              for (int i = 0; i < MH; ++i)
                before[i] = __builtin_bit_cast(f32x4_v, __builtin_amdgcn_raw_buffer_load_b128(slot, own + (quad * kQuad + (half * MH + i) * 8192), 0, kThrough));
#pragma unroll
              for (int i = 0; i < MH; ++i) acc[quad >> 1][quad & 1][half * MH / 2 + i / 2][i % 2] += before[i];
              __builtin_amdgcn_sched_barrier(0);
            }
          }
          if (!whole) {
#pragma unroll
            for (int i = 0; i < 2 * MH; ++i)
              __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_v, acc[quad >> 1][quad & 1][i / 2][i % 2]), slot,
                                                     own + (quad * kQuad + i * 8192), 0, kThrough);
          }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // they are in memory before they are asked for
        if (!whole) {
          more = next_segment(cc, tile, k0, k1);
          continue;
        }
      }
    }
    if (whole) {
      int which, m0, n0;
      locate(tile, which, m0, n0);
      const GemmEpilogue& e = p.q[which].ep;
      const int ln = hidden_lane(), kind = epilogue_kind(e, m0, BM);
      const int m = m0 + wm * (16 * MH) + (ln & 15), n = n0 + wn * 32 + (ln >> 4) * 8;
      const bool heads = has_heads(which);
      if (!heads) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int h = 0; h < 2; ++h) finish_quadrant<T, MH, HEADS, APART>(kind, e, m0, m + h * HM, n + b * 128, acc[h][b]);
      }
      // (behind the other, and opaque to it: what comes first keeps the sums in their registers whichever is taken)
      if constexpr (HEADS) {
        if (scalar(heads) != 0) finish_heads(p.heads[which], e, m0, n0, ln);
      }
    } else if constexpr (!APART) {
      // A part of a cut tile. The parts share the tile's four quadrants out between them: part i adds up and finishes quadrants i,
      // i + parts, ..., which it keeps in LDS (each thread its own accumulators; no tile load is in flight any more), and
      // leaves the others in its slot.
      // (a vector instruction right behind a 16-byte store must not write the store's data registers. The compiler puts the wait
      // there, but takes a store with an offset in a scalar register for safe, and accumulators of the last lanes went to memory
      // overwritten now and then. So the slot is in the descriptor, the rest in the vector offset, and no store has a scalar one.)
      const auto slot = __builtin_amdgcn_make_buffer_rsrc(p.slots + static_cast<int64_t>(v) * kTileSlot, 0, kTileSlot, 0x00020000);
      const uint32_t own = static_cast<uint32_t>((wave * 64 + hidden_lane()) * 16);
      const int mine = quadrants();
#pragma unroll
      for (int quad = 0; quad < 4; ++quad) {
        if (mine >> quad & 1) continue;
#pragma unroll
        for (int i = 0; i < 2 * MH; ++i)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_v, acc[quad >> 1][quad & 1][i / 2][i % 2]), slot,
                                                 own + (quad * kQuad + i * 8192), 0, kThrough);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the pieces have reached memory before the ticket is taken
      __syncthreads();
      if (tid == 0) {
        unsigned long long* word = p.counters + (tile - p.whole);
        // two atomics of one thread on one address: applied in program order
        __hip_atomic_fetch_max(word, p.epoch << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned old = static_cast<unsigned>(__hip_atomic_fetch_add(word, kArrival, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        flag[1] = (old & 15u) + 1 == static_cast<unsigned>(p.parts) ? old >> 4 & 15u : 0;  // the last to arrive: what was given up
      }
      int at = 0;
#pragma unroll
      for (int quad = 0; quad < 4; ++quad) {
        if (!(mine >> quad & 1)) continue;
#pragma unroll
        for (int i = 0; i < 2 * MH; ++i) *reinterpret_cast<f32x4_v*>(lds + at + own + i * 8192) = acc[quad >> 1][quad & 1][i / 2][i % 2];
        at = scalar(at + kQuad);
      }
    }
    more = next_segment(cc, tile, k0, k1);
  }
  if (!APART && has_part) {
    // A part looks for all parts of its tile to have arrived, a bounded number of times; then it gives its quadrants up (which fails
    // if the last one has arrived by now) and leaves them to the last to arrive.
    const int part = quotient(v, cut), t = v - part * cut, parts = p.parts, mine = quadrants();
    unsigned long long* word = p.counters + t;
    const unsigned all = static_cast<unsigned>(parts);
    const auto slots = __builtin_amdgcn_make_buffer_rsrc(p.slots, 0, G * kTileSlot, 0x00020000);
    if (tid == 0) {
      int got = 0;
      for (int look = 0; look < kLooks && got == 0 && mine != 0; ++look) {
        const unsigned w = static_cast<unsigned>(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if ((w & 15u) == all) got = mine;
        else __builtin_amdgcn_s_sleep(8);
      }
      flag[0] = got;
    }
    __syncthreads();
    int got = scalar(flag[0]);
    if (got == 0) {
      const auto slot = __builtin_amdgcn_make_buffer_rsrc(p.slots + static_cast<int64_t>(v) * kTileSlot, 0, kTileSlot, 0x00020000);
      const uint32_t own = static_cast<uint32_t>((wave * 64 + hidden_lane()) * 16);
      int at = 0;
      for (int left = mine; left != 0; left &= left - 1) {
        const int quad = __builtin_ctz(left);
#pragma unroll
        for (int i = 0; i < 2 * MH; ++i)
          __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4_v*>(lds + at + own + i * 8192), slot,
                                                 own + (quad * kQuad + i * 8192), 0, kThrough);
        at = scalar(at + kQuad);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // (and the flag has been read)
      if (tid == 0) {
        const unsigned old = static_cast<unsigned>(__hip_atomic_fetch_or(word, static_cast<unsigned long long>(mine) << 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        flag[0] = (old & 15u) == all ? mine : 0;
      }
      __syncthreads();
      got = scalar(flag[0]);
    }
    got = scalar(got | flag[1]);
    int which, m0, n0;
    locate(p.whole + t, which, m0, n0);
    const GemmEpilogue& e = p.q[which].ep;
    const int kind = epilogue_kind(e, m0, BM);
    for (; got != 0; got &= got - 1) {
      const int quad = __builtin_ctz(got);
      const bool kept = mine >> quad & 1;
      const int ln = hidden_lane();
      const uint32_t off = static_cast<uint32_t>((wave * 64 + ln) * 16 + quad * kQuad);
      const uint32_t kept_at = static_cast<uint32_t>((wave * 64 + ln) * 16) + ((mine & ((1 << quad) - 1)) != 0 ? kQuad : 0);
      f32x4_v sum[MH][2];
      // all parts of the quadrant in one round trip, added in the order of the parts
      auto add_up = [&](auto pc) __attribute__((always_inline)) {
        constexpr int P = decltype(pc)::value;
        f32x4_v r[P][2 * MH];
#pragma unroll
        for (int j = 0; j < P; ++j) {
          if (kept && j == part) {
#pragma unroll
            for (int i = 0; i < 2 * MH; ++i) r[j][i] = *reinterpret_cast<const f32x4_v*>(lds + kept_at + i * 8192);
          } else {
#pragma unroll
            for (int i = 0; i < 2 * MH; ++i)
              r[j][i] = __builtin_bit_cast(f32x4_v, __builtin_amdgcn_raw_buffer_load_b128(slots, off + i * 8192, (t + j * cut) * kTileSlot, kThrough));
          }
        }
#pragma unroll
        for (int i = 0; i < 2 * MH; ++i) {
          sum[i / 2][i % 2] = r[0][i];
#pragma unroll
          for (int j = 1; j < P; ++j) sum[i / 2][i % 2] += r[j][i];
        }
      };
      if (parts == 2) add_up(std::integral_constant<int, 2>{});
      else if (parts == 3) add_up(std::integral_constant<int, 3>{});
      else if (MH > 2 || parts == 4) add_up(std::integral_constant<int, 4>{});
      else if constexpr (MH <= 2) {
        if (parts == 5) add_up(std::integral_constant<int, 5>{});
        else if (parts == 6) add_up(std::integral_constant<int, 6>{});
        else if (parts == 7) add_up(std::integral_constant<int, 7>{});
        else add_up(std::integral_constant<int, 8>{});
      }
      const int r = (quad >> 1) * HM + wm * (16 * MH) + (ln & 15), n = n0 + (quad & 1) * 128 + wn * 32 + (ln >> 4) * 8;
      if (has_heads(which)) {  // (the same in all wavefronts)
        if constexpr (HEADS) {
          const HeadsOut& hd = p.heads[which];
          const int third = quotient(n0 + (quad & 1) * 128 + wn * 32, hd.HD), d = n & (hd.D - 1);
          u32x4 bias = {0u, 0u, 0u, 0u}, weight = bias;
          if (e.bias != nullptr && third < 3) bias = load_raw(static_cast<const T*>(e.bias) + n);
          if (third < 2) weight = load_raw(static_cast<const T*>(third == 0 ? hd.wq : hd.wk) + d);
          HeadRows<MH> rows;
          rows.ask(hd, e.M, m0, r, d);
          loads_arrived();
          float* const sq = squares + (quad & 1) * BM * 4;
          u32x4 x[MH];
          square_heads<T, MH>(sum, bias, x, sq, r, wn, ln >> 4);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          barrier();
          if (third < 3) store_heads<T, MH>(hd, x, rows, sq, r, wn, third, n, weight);
        }
      } else {
        finish_quadrant<T, MH, HEADS, APART>(kind, e, m0, m0 + r, n, sum);
      }
    }
    // the last to leave hands the word back at zero
    if (tid == 0 && ((__hip_atomic_fetch_add(word, kDeparture, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 8) & 15u) + 1 == all)
      __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS outlives the workgroup
}

int row_tiles(int M, int bm) { return (M + bm - 1) / bm; }

// What a launch of `plan` takes beside its heads.
// Rows of padding are fetched from where they would lie: past the end of the operand, for which its descriptor answers zeros. A tile of 256 rows
// is bound by power, and a product of zeros takes little; copies of the last row stood in their place. Alone (us, copies / zeros): 8192 + 300
// rows, N=9216, K=3072, 355.0 / 350.7; 2706 rows, 5120 x 5120, 109.2 / 108.2; 512 + 80 rows, N=9216, tiles of 128 rows, 57.8 / 58.5. In whole
// models those of 128 rows gain a little too (two prompts of 171 and 23 at 1024 rows, eight blocks, 4693 / 4682, else the same), those of 256
// more: 950 + 12 rows, five blocks, 2768 / 2732; 6156 + 44, six, 19714 / 19305; 169 + 121 and 269, five, 1811 / 1731.
// Offsets have 32 bits: an operand whose padding would wrap around keeps the copies.
inline void fill_tile_params(TileParams& p, const TilePlan& plan, const GemmCall* c, int count, const TileX2* x2, void* scratch) {
  for (int i = 0; i < 3; ++i) {
    const GemmCall& g = c[i < count ? i : 0];
    TileProblem& q = p.q[i];
    q.x = g.x; q.w = g.w; q.M = g.M; q.N = g.N;
    q.ldx = static_cast<uint32_t>(g.ldx * 2); q.ldw = static_cast<uint32_t>(g.ldw * 2);
    const int k1 = x2 ? x2->k_split : g.K;
    q.x2 = x2 ? x2->x : g.x;
    q.ldx2 = x2 ? static_cast<uint32_t>(x2->ldx * 2) : q.ldx;
    q.k_split = k1 / kTileK;
    q.x_bytes = static_cast<uint32_t>((static_cast<uint64_t>(g.M - 1) * g.ldx + k1) * 2);
    q.x2_bytes = x2 ? static_cast<uint32_t>((static_cast<uint64_t>(g.M - 1) * x2->ldx + g.K - k1) * 2) : q.x_bytes;
    q.w_bytes = static_cast<uint32_t>((static_cast<uint64_t>(g.N - 1) * g.ldw + g.K) * 2);
    q.m_tiles = (g.M + plan.bm - 1) / plan.bm;
    q.n_tiles = (g.N + kTileN - 1) / kTileN;
    q.x_last = tile_padding_row(g.M, plan.bm, x2 ? std::max(g.ldx, x2->ldx) : g.ldx, g.K);
    q.w_last = tile_padding_row(g.N, kTileN, g.ldw, g.K);
    q.ep = gemm_epilogue_of(g);
  }
  p.tiles0 = plan.tiles0; p.tiles1 = plan.tiles1; p.tiles = plan.tiles; p.whole = plan.whole; p.parts = plan.parts;
  p.k_steps = c[0].K / kTileK;
  p.counters = static_cast<unsigned long long*>(scratch);
  p.epoch = plan.parts > 1 ? next_ticket_epoch() : 0;
  p.slots = scratch ? static_cast<char*>(scratch) + kGemmCounterBytes : nullptr;
}

}  // namespace

}  // namespace odit
