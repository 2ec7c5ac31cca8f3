// 16-bit GEMM y = x W^T for one problem, or two of the same N and K in ONE launch (the image and the text rows of a
// dual-stream block: different weights, the same widths), where one tile per workgroup leaves CUs idle or badly balanced.
//
// Work split ("stream-K"): the output of each problem is cut into BM x BN tiles and every tile's reduction into steps
// of 64 elements. The workgroups come in groups of m_tiles (one per row tile of either problem); the steps of all
// feature tiles, laid end to end, are dealt out in equal contiguous ranges to the groups, so that every CU has the same
// number of steps whatever the shapes. The workgroups of a group sit on one XCD and walk the same (feature tile, step)
// pairs side by side: a piece of W comes from memory once and is found in that XCD's L2 by the others. A range covers the
// tail of one feature tile, maybe whole tiles, and the head of another. A tile finished by one workgroup alone goes
// straight through the epilogue. Otherwise a contributor that finds the tile's counter short of full leaves its fp32
// partial tile in a scratch slot (write-through stores) and takes a ticket; the last arriver adds the partial tiles in
// workgroup order (its own, still in registers, in its place: the sum does not depend on who arrives last), runs the
// epilogue and resets the counter. Nobody waits for anybody. A ticket word is (epoch << 16 | tickets): a contributor first
// raises the word to this launch's epoch with an atomic maximum, so what an earlier launch left there (one that never
// finished, say) cannot be mistaken for this launch's tickets.
//
// Workgroup: 8 wavefronts = 2 halves of each step's reduction x 4 corners of the tile (2 x 2 of 64 x BN / 2; BM = 64: 4
// side by side of 64 x BN / 4), v_mfma_f32_32x32x16 with W rows as the A operand and x rows as B: a lane ends up with one
// row m of the output and 4 x 4 consecutive features n per accumulator. When the range ends the two halves meet through
// LDS, each wave keeping half of the accumulators.
//
// Tile movement: a pipeline step is a BM x 64 piece of x and a BN x 64 piece of W, 128-byte rows, moved from global
// memory straight into LDS by `buffer_load_dwordx4 ... lds` (one wave instruction fills 1 KB = 8 rows; lane l's 16 bytes
// land at base + 16 l, so the lane chooses WHAT to fetch: the 16-byte chunk (l % 8) ^ ((row >> 1) & 7) of its row, which
// makes the 16-byte fragment reads of 16 consecutive rows cover all 64 banks). As many LDS stages as 160 KB hold (3 to 6).
//
// Pipeline: a wave multiplies two k16 slices per step. One barrier per step, BETWEEN the slices: in front of it a wave
// has the second slice's fragments in registers and its own loads of the next step have landed, so behind it this step's
// stage is free and the next stage is complete, and the next step's first fragments are read while the second slice is
// multiplied.
//
// What bounds it. 0.70 us per 128 x 192 x 64 step at M=1024 (1.15 PFLOP/s while the main loop runs), 0.81 at M=512, with
// 3 stages or 4, at any row stride of the operands: 40 KB per step and CU out of L2, 46 to 57 GB/s per CU (98 is what a
// bare loop of such loads reaches), and 120 KB through LDS for 768 cycles of matrix work. Around the loop a launch costs 8
// us (cold first loads, halves meeting, epilogue), each hand-over of a partial tile 2 to 8: ranges are laid so that few
// happen (plan_streamk). Measured, cold weights, us, beside the library's first choice: M=80 and N=9216, K=3072 21.0 / 28.0;
// N=3072, K=12288 31 / 57; M=512 and N=9216 42.6 / 41.9; N=3072, K=12288 52 / 69. Both streams of a block of a 256-pixel
// image (512 + 80 rows) in one launch, against two library launches: QKV 42 / 70, MLP down 61 / 127.
#include <type_traits>

#include "gemm_epilogue.h"

namespace odit {

namespace {

constexpr int kWaves = 8;

struct GemmProblem {
  const void *x, *w;
  int M;
  int64_t ldx, ldw;
  GemmEpilogue ep;
  uint32_t x_bytes, w_bytes;
};

struct GemmParams {
  GemmProblem p0, p1;
  int N, k_steps;
  int mt0, m_tiles;      // row tiles of the first problem, of both
  int workers, groups;
  unsigned total_steps;  // per group: feature tiles x reduction steps
  unsigned long long* counters;  // one ticket word per output tile: (epoch << 16 | tickets drawn), zero between launches
  unsigned long long epoch;      // larger than that of any earlier launch of the process
  char* slots;
};

typedef __attribute__((address_space(3))) void* lds_void_p;

// worker whose range [v S / W, (v + 1) S / W) holds `step` (the launcher keeps (S + 1) W below 2^32)
__device__ __forceinline__ int worker_of(unsigned step, unsigned S, unsigned W) {
  return static_cast<int>(((step + 1) * W - 1) / S);
}
__device__ __forceinline__ const char* uniform(const char* p) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  const uint64_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a)) & 0xffffffffull;
  const uint64_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32)) & 0xffffffffull;
  return reinterpret_cast<const char*>(lo | (hi << 32));
}

// 16 bytes per lane past the XCD's L2, where the workgroups of all XCDs see them (what an agent-scope atomic store and
// load of a word do, four words at a time); `base` is wave-uniform, `off` the lane's byte offset. The address may come
// out of a v_readfirstlane right in front: a memory instruction may read a scalar register 5 wait states after a vector
// instruction has written it and no sooner, and the compiler does not look into these statements, so they wait themselves; and a
// vector instruction may write a 16-byte store's data registers 2 wait states behind it and no sooner.
__device__ __forceinline__ void store_through(const char* base, uint32_t off, f32x4_v v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc1\n\ts_nop 1" ::"v"(off), "v"(v), "s"(base) : "memory");
#endif
}
// N vectors 1 KB apart in one round trip (loads and wait in one statement: nothing can touch the registers before the
// data is there)
template <int N> __device__ __forceinline__ void load_through(f32x4_v (&v)[N], const char* base, uint32_t off) {
  static_assert(N == 4 || N == 8 || N == 12 || N == 16, "whole 4 KB runs");
#if defined(__HIP_DEVICE_COMPILE__)
#define ODIT_RUN(a, b, c, d, s)                                                                          \
  "global_load_dwordx4 %" #a ", %[o], %[" #s "] sc1\n\tglobal_load_dwordx4 %" #b ", %[o], %[" #s "] offset:1024 sc1\n\t" \
  "global_load_dwordx4 %" #c ", %[o], %[" #s "] offset:2048 sc1\n\tglobal_load_dwordx4 %" #d ", %[o], %[" #s "] offset:3072 sc1\n\t"
  if constexpr (N == 4) {
    asm volatile("s_nop 4\n\t" ODIT_RUN(0, 1, 2, 3, s0) "s_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                 : [o] "v"(off), [s0] "s"(base)
                 : "memory");
  } else if constexpr (N == 8) {
    asm volatile("s_nop 4\n\t" ODIT_RUN(0, 1, 2, 3, s0) ODIT_RUN(4, 5, 6, 7, s1) "s_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
                 : [o] "v"(off), [s0] "s"(base), [s1] "s"(base + 4096)
                 : "memory");
  } else if constexpr (N == 12) {
    asm volatile("s_nop 4\n\t" ODIT_RUN(0, 1, 2, 3, s0) ODIT_RUN(4, 5, 6, 7, s1) ODIT_RUN(8, 9, 10, 11, s2) "s_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
                   "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
                 : [o] "v"(off), [s0] "s"(base), [s1] "s"(base + 4096), [s2] "s"(base + 8192)
                 : "memory");
  } else {
    asm volatile("s_nop 4\n\t" ODIT_RUN(0, 1, 2, 3, s0) ODIT_RUN(4, 5, 6, 7, s1) ODIT_RUN(8, 9, 10, 11, s2) ODIT_RUN(12, 13, 14, 15, s3) "s_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
                   "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11]), "=&v"(v[12]), "=&v"(v[13]), "=&v"(v[14]), "=&v"(v[15])
                 : [o] "v"(off), [s0] "s"(base), [s1] "s"(base + 4096), [s2] "s"(base + 8192), [s3] "s"(base + 12288)
                 : "memory");
  }
#undef ODIT_RUN
#endif
}

// BM x BN: rows of x and features per tile (128 x 256, 128 x 192, 128 x 128 or 64 x 128)
template <typename T, int BM, int BN>
__global__ __launch_bounds__(kWaves * 64, 1) void gemm_streamk_kernel(const GemmParams p) {
  using M = Mma<T>;
  using frag = typename M::frag;
  constexpr int WM = BM / 64;                 // corners along the rows
  constexpr int TM = 2, TN = BN * WM / 128;   // 32 x 32 accumulators of a corner
  constexpr int ACC = TM * TN, OWN = ACC / 2;
  constexpr int kXBytes = BM * kGemmBK * 2;
  constexpr int kStage = kXBytes + BN * kGemmBK * 2;
  constexpr int kStages = 160 * 1024 / kStage;  // 6, 5, 4 or 3: what the LDS of a CU holds
  constexpr int kInst = kStage / 1024, kIPW = kInst / kWaves, kXInst = kXBytes / 1024;
  constexpr int H0 = (kIPW + 1) / 2;          // tile-load instructions that go out with the second slice
  static_assert(kInst % kWaves == 0, "tile loads must divide evenly over the wavefronts");
  constexpr int kPitch = TN * 32 + 4;         // floats per staged output row
  constexpr int kEpiBytes = 4 * 64 * kPitch * 4;
  constexpr int kLds = kStages * kStage > kEpiBytes ? kStages * kStage : kEpiBytes;
  __shared__ __attribute__((aligned(1024))) char lds[kLds];
  int* const flag = reinterpret_cast<int*>(lds + kLds - 16);  // behind what the exchange and the epilogue use
  static_assert(kWaves * OWN * 4096 + 16 <= kLds && kEpiBytes + 16 <= kLds, "the flag must not be written over");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, kept in a scalar register
  const int l32 = lane & 31, hh = lane >> 5;
  const int kh = wave >> 2, w4 = wave & 3;  // half of each step's reduction, corner of the tile
  const int wm = WM == 2 ? (w4 & 1) : 0, wn = WM == 2 ? (w4 >> 1) : w4;
  const int lrow = lane >> 3, lpc = lane & 7;

  const int v = xcd_remap(blockIdx.x, p.workers);
  const int group = v / p.m_tiles, mt = v - group * p.m_tiles;
  const bool second = mt >= p.mt0;
  const GemmProblem& q = second ? p.p1 : p.p0;
  const unsigned S = p.total_steps, G = p.groups;
  unsigned s = group * S / G;
  const unsigned s_end = (group + 1) * S / G;

  auto make_rsrc = [](const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    u32x4_v r;
    r.x = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    r.y = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32) & 0xffffu);
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;
    return r;
  };
  const u32x4_v xrsrc = make_rsrc(q.x, q.x_bytes);
  const u32x4_v wrsrc = make_rsrc(q.w, q.w_bytes);
  const int m0 = (second ? mt - p.mt0 : mt) * BM;
  // instruction i of this wave's share of a step is number wave * kIPW + i: it fills 1 KB of the stage, x first
  const int q0 = wave * kIPW;

  // fragment (sub-tile t, k16 slice kq of this wave's half) of a piece: row 32 t + l32, logical chunk 2 (2 kh + kq) + hh
  const int frag0 = l32 * 128 + (((4 * kh + hh) ^ ((l32 >> 1) & 7)) << 4);
  // The halves of the reduction share a corner's accumulators out between them at the end: the first OWN registers of a
  // wave are the ones it keeps, so the wave of the second half starts half a corner further (along the features, or
  // along the rows where a corner is one accumulator wide).
  constexpr bool kAlongN = TN % 2 == 0;
  constexpr int kFar = (kAlongN ? TN : TM) / 2 * (32 * 128);  // half a corner in LDS bytes
  const int near = kh ? kFar : 0, away = kh ? -kFar : 0;      // for the registers of the first half, of the second
  const int xf0 = wm * (64 * 128) + frag0, wf0 = kXBytes + wn * (TN * 32 * 128) + frag0;

  while (s < s_end) {
    const int t = static_cast<int>(s / static_cast<unsigned>(p.k_steps));  // feature tile
    const int kk0 = static_cast<int>(s) - t * p.k_steps;
    const int left = static_cast<int>(s_end - s);
    const int nk = p.k_steps - kk0 < left ? p.k_steps - kk0 : left;
    const int n0 = t * BN;

    // per-lane byte offsets of the chunks this lane moves (rows past the end re-read the last row:
    // their products land in output rows / features that are never stored)
    uint32_t voff[kIPW];
#pragma unroll
    for (int i = 0; i < kIPW; ++i) {
      const bool isx = q0 + i < kXInst;
      const int r = (isx ? q0 + i : q0 + i - kXInst) * 8 + lrow;
      int rg = isx ? m0 + r : n0 + r;
      const int last = isx ? q.M - 1 : p.N - 1;
      rg = rg < last ? rg : last;
      voff[i] = static_cast<uint32_t>(rg) * static_cast<uint32_t>((isx ? q.ldx : q.ldw) * 2) +
                static_cast<uint32_t>((lpc ^ ((r >> 1) & 7)) << 4);
    }
    // instruction i of this wave's share of step kk's tile loads
    auto issue1 = [&](int kk, int stage, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
      const uint32_t soff = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(kk) * (kGemmBK * 2));
      const uint32_t dst = __builtin_amdgcn_readfirstlane(
          static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_p)(lds + stage * kStage + (q0 + i) * 1024))));
      const u32x4_v rs = q0 + i < kXInst ? xrsrc : wrsrc;  // wave-uniform
      load_lds16(dst, voff[i], rs, soff);
#endif
    };

    f32x16_v acc[ACC];  // blocks (tn, tm) of the corner, those of a half together
#pragma unroll
    for (int a = 0; a < ACC; ++a)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][e] = 0.f;

    frag xf[2][TM], wf[2][TN];
    // fragment number f (x first) of slice kq of the step in `stage`
    auto read1 = [&](int stage, int kq, int f) {
      const char* b = lds + stage * kStage;
      if (f < TM) {
        const int shift = kAlongN ? 0 : (f < TM / 2 ? near : away);
        xf[kq][f] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(b + shift + f * (32 * 128) + (xf0 ^ (kq * 32))));
      } else {
        const int shift = !kAlongN ? 0 : (f - TM < TN / 2 ? near : away);
        wf[kq][f - TM] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(b + shift + (f - TM) * (32 * 128) + (wf0 ^ (kq * 32))));
      }
    };
    // the matrix instructions of slice kq, with the reads of the other slice's fragments (from `stage`) and `n` tile-load
    // instructions i0.. of step kk (into `ld_stage`) in between
    auto slice = [&](int kq, int stage, bool load, int kk, int ld_stage, auto i0c, auto nc) {
      constexpr int i0 = decltype(i0c)::value, n = decltype(nc)::value;
#pragma unroll
      for (int a = 0; a < ACC; ++a) {
        acc[a] = M::run(wf[kq][kAlongN ? a / TM : a % TN], xf[kq][kAlongN ? a % TM : a / TN], acc[a]);
        if (a < TM + TN) read1(stage, kq ^ 1, a);
        if (a + 1 == ACC)
#pragma unroll
          for (int f = ACC; f < TM + TN; ++f) read1(stage, kq ^ 1, f);
#pragma unroll
        for (int i = 0; i < n; ++i)
          if (i * ACC / n == a && load) issue1(kk, ld_stage, i0 + i);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    using std::integral_constant;

    __syncthreads();  // every wave has left the LDS uses of the previous range
    // loads of the first kStages steps (of the last of them: the first part)
    auto prologue = [&](auto self, auto dc) -> void {
      constexpr int d = decltype(dc)::value;
      if (d < nk) {
#pragma unroll
        for (int i = 0; i < (d + 1 < kStages ? kIPW : H0); ++i) issue1(kk0 + d, d, i);
        if constexpr (d + 1 < kStages) self(self, integral_constant<int, d + 1>{});
      }
    };
    prologue(prologue, integral_constant<int, 0>{});
    // step 0 has landed when at most the later steps' loads are in flight
    if (nk >= kStages) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 2) * kIPW + H0) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int f = 0; f < TM + TN; ++f) read1(0, 0, f);
    int st = 0;  // stage of step i
    for (int i = 0; i < nk; ++i) {
      const int st_next = st + 1 == kStages ? 0 : st + 1, st_last = st == 0 ? kStages - 1 : st - 1;
      // first slice; the rest of step i + kStages - 1's tile loads
      slice(0, st, i + kStages - 1 < nk, kk0 + i + kStages - 1, st_last, integral_constant<int, H0>{}, integral_constant<int, kIPW - H0>{});
      // the second slice's fragments are in registers and this wave's loads of step i + 1 have landed (those of later
      // steps may be in flight) ...
      if (i + kStages - 1 < nk) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kStages - 2) * kIPW) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      }
      // ... in every wave: this step's stage is free, the next one is complete
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      // second slice; the first loads of step i + kStages (after the last step this reads a stage that nobody has filled:
      // the values are never used)
      slice(1, st_next, i + kStages < nk, kk0 + i + kStages, st, integral_constant<int, 0>{}, integral_constant<int, H0>{});
      st = st_next;
    }
    s += nk;

    // ---- the two halves of the reduction meet: a wave keeps its first OWN accumulators (blocks OWN kh + 0 .. OWN - 1 of
    // the corner), gives the others to its partner through LDS and adds the partner's to its own ----
    f32x16_v own[OWN];
    // (the lane's numbers are hidden from the compiler from here on: it would form every address below once in front of
    // all ranges and keep them in registers that the main loop needs)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    {
      __syncthreads();  // the stages are idle from here
      f32x4_v* xch = reinterpret_cast<f32x4_v*>(lds);  // [w4][giver kh][OWN][4 g][64 lanes] x 16 bytes
      auto part = [&](int sl, int g, int giver) -> f32x4_v& { return xch[(((w4 * 2 + giver) * OWN + sl) * 4 + g) * 64 + ln]; };
#pragma unroll
      for (int sl = 0; sl < OWN; ++sl)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4_v r;
#pragma unroll
          for (int u = 0; u < 4; ++u) r[u] = acc[OWN + sl][g * 4 + u];
          part(sl, g, kh) = r;
        }
      __syncthreads();
#pragma unroll
      for (int sl = 0; sl < OWN; ++sl)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4_v r = part(sl, g, kh ^ 1);
#pragma unroll
          for (int u = 0; u < 4; ++u) own[sl][g * 4 + u] = acc[sl][g * 4 + u] + r[u];
        }
    }

    // ---- who else works on this tile ----
    const unsigned tile_s0 = static_cast<unsigned>(t) * p.k_steps;
    const int v_first = worker_of(tile_s0, S, G);  // first and last group on this feature tile
    const int v_last = worker_of(tile_s0 + p.k_steps - 1, S, G);
    if (v_first != v_last) {
      // slot 0 of a workgroup is for the tile its range starts in, slot 1 for any later one;
      // layout of a slot: [w4][kh][OWN][4 g][64 lanes] x 16 bytes
      auto slot_of = [&](int j) {
        const int first_tile = static_cast<int>((j * S / G) / static_cast<unsigned>(p.k_steps));
        return uniform(p.slots + static_cast<size_t>(2 * (j * p.m_tiles + mt) + (first_tile == t ? 0 : 1)) * kGemmSlotBytes +
               static_cast<size_t>((w4 * 2 + kh) * OWN * 4096));
      };
      const uint32_t lane_off = ln * 16;
      unsigned long long* ctr = p.counters + t * p.m_tiles + mt;
      const unsigned long long full = (p.epoch << 16) + static_cast<unsigned>(v_last - v_first);
      // When every other contributor has already taken its ticket this workgroup is the last arriver
      // and keeps its partial tile in registers; otherwise the tile goes to the slot first and the
      // ticket is taken after it (whoever then holds the last ticket reduces).
      if (tid == 0)
        *reinterpret_cast<volatile int*>(flag) =
            __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == full ? 1 : 0;
      __syncthreads();
      const bool known_last = __builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(flag)) != 0;
      __syncthreads();  // the flag is read before it is written again
      if (known_last) {
        if (tid == 0) __hip_atomic_store(ctr, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        const char* mine = slot_of(group);
#pragma unroll
        for (int sl = 0; sl < OWN; ++sl)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4_v r;
#pragma unroll
            for (int u = 0; u < 4; ++u) r[u] = own[sl][g * 4 + u];
            store_through(mine + (sl * 4 + g) * 1024, lane_off, r);
          }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the partial tile has reached memory before the ticket is taken
        __syncthreads();
        if (tid == 0) {
          // two atomics of one thread on one address: applied in program order
          __hip_atomic_fetch_max(ctr, p.epoch << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const unsigned long long ticket = __hip_atomic_fetch_add(ctr, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const int last = ticket == full;
          if (last) __hip_atomic_store(ctr, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          *reinterpret_cast<volatile int*>(flag) = last;
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(flag)) == 0) continue;
      }
      // last arriver: partial tiles in workgroup order (its own, still in registers, in its place), one
      // contributor per round trip
      f32x16_v sum[OWN];
#pragma unroll
      for (int sl = 0; sl < OWN; ++sl)
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[sl][e] = 0.f;
      for (int j = v_first; j <= v_last; ++j) {
        if (j == group) {
#pragma unroll
          for (int sl = 0; sl < OWN; ++sl)
#pragma unroll
            for (int e = 0; e < 16; ++e) sum[sl][e] += own[sl][e];
        } else {
          f32x4_v r[OWN * 4];
          load_through(r, slot_of(j), lane_off);
#pragma unroll
          for (int sl = 0; sl < OWN; ++sl)
#pragma unroll
            for (int e = 0; e < 16; ++e) sum[sl][e] += r[sl * 4 + (e >> 2)][e & 3];
        }
      }
#pragma unroll
      for (int sl = 0; sl < OWN; ++sl) own[sl] = sum[sl];
    } else {
      __syncthreads();  // the exchange area is read out before the epilogue reuses it
    }

    // ---- epilogue ----
    // A lane holds one output row and 4 x 4 features per accumulator: stored from there, every wave
    // instruction would touch 32 output rows with 16 bytes each. Each corner goes through LDS instead (fp32, padded
    // rows: the 16-byte writes of 16 rows cover all banks) and leaves as 16-byte pieces of 8 features, consecutive
    // lanes on one output row; bias, activation, gate and residual are applied on the way out, where their loads
    // are row-contiguous too.
    {
      float* stg = reinterpret_cast<float*>(lds) + w4 * (64 * kPitch);
#pragma unroll
      for (int sl = 0; sl < OWN; ++sl) {
        const int a = kh * OWN + sl, tn = kAlongN ? a / TM : a % TN, tm = kAlongN ? a % TM : a / TN;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4_v r;
#pragma unroll
          for (int u = 0; u < 4; ++u) r[u] = own[sl][g * 4 + u];
          *reinterpret_cast<f32x4_v*>(stg + (tm * 32 + (ln & 31)) * kPitch + tn * 32 + g * 8 + (ln >> 5) * 4) = r;
        }
      }
      __syncthreads();  // a corner is written by two waves and read by the same two
      constexpr int CPR = TN * 4;              // 16-byte output pieces per row of the corner
      constexpr int IT = CPR / 2;              // per lane of each of the two waves
#pragma unroll 4
      for (int it = 0; it < IT; ++it) {
        const int idx = (kh * IT + it) * 64 + ln;
        const int row = idx / CPR, ch = idx % CPR;
        const int m = m0 + wm * 64 + row;
        const int n = n0 + wn * (TN * 32) + ch * 8;
        const f32x4_v lo = *reinterpret_cast<const f32x4_v*>(stg + row * kPitch + ch * 8);
        const f32x4_v hi = *reinterpret_cast<const f32x4_v*>(stg + row * kPitch + ch * 8 + 4);
        if (m >= q.M || n >= p.N) continue;
        float y[8];
#pragma unroll
        for (int u = 0; u < 4; ++u) { y[u] = lo[u]; y[4 + u] = hi[u]; }
        gemm_epilogue_store8<T>(q.ep, m, n, y);
      }
    }
  }
}

GemmProblem problem_of(const GemmCall& c) {
  GemmProblem q;
  q.x = c.x; q.w = c.w; q.M = c.M; q.ldx = c.ldx; q.ldw = c.ldw;
  q.ep = gemm_epilogue_of(c);
  q.x_bytes = static_cast<uint32_t>((static_cast<uint64_t>(c.M - 1) * c.ldx + c.K) * 2);
  q.w_bytes = static_cast<uint32_t>((static_cast<uint64_t>(c.N - 1) * c.ldw + c.K) * 2);
  return q;
}

int row_tiles(int M, int bm) { return (M + bm - 1) / bm; }

}  // namespace

int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cus[dev] = n;
  }
  return cus[dev];
}

// whether the kernel can run one problem
bool gemm_streamk_takes(const GemmCall& c, int dtype) {
  if (dtype != ODIT_BF16 && dtype != ODIT_F16) return false;
  if (c.M < 1 || c.K < kGemmBK || c.K % kGemmBK != 0 || c.N % 8 != 0) return false;
  if (c.ldx % 8 != 0 || c.ldw % 8 != 0 || c.ldo % 8 != 0) return false;
  if (!aligned16(c.x) || !aligned16(c.w) || !aligned16(c.out)) return false;
  if (c.bias != nullptr && (reinterpret_cast<uintptr_t>(c.bias) & 15u) != 0) return false;
  const bool gated = c.epilogue == ODIT_EPI_GATED_RESIDUAL || c.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
  if (gated) {
    if (c.residual == nullptr || c.ldr % 8 != 0 || !aligned16(c.residual)) return false;
    if (c.gate != nullptr && (!aligned16(c.gate) || c.ldg % 8 != 0)) return false;
    if (c.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE && !c.gate_f32) return false;
  }
  const uint64_t xb = (static_cast<uint64_t>(c.M - 1) * c.ldx + c.K) * 2, wb = (static_cast<uint64_t>(c.N - 1) * c.ldw + c.K) * 2;
  if (xb >= (1ull << 32) || wb >= (1ull << 32)) return false;
  return static_cast<int64_t>(row_tiles(c.M, 64)) * ((c.N + 127) / 128) * 8 <= static_cast<int64_t>(kGemmCounterBytes) &&
         row_tiles(c.M, 64) <= kGemmMaxWorkers &&
         (static_cast<int64_t>((c.N + 127) / 128) * (c.K / kGemmBK) + 1) * kGemmMaxWorkers < (1ll << 32);
}

// How a launch is cut: tile shape, and groups of workgroups over the feature tiles. With G a multiple of the feature tiles
// every range lies inside one tile, which is reduced over G / n_tiles workgroups (one range, at most one partial tile to
// hand over); with as many groups as there are CUs for, ranges run on across tile boundaries: fewer steps each, but two
// partial tiles per workgroup. The times are fitted to 16 <= M <= 1024 rows of the four projections of width 3072 (us; a
// step of 64: 128-wide tiles 0.62, 192 0.74, 256 0.88; a launch 8; each further contributor of a tile 1.2, 2.0, 2.7; a
// second range 4, 10, 16; a further whole tile 6). M=512, N=9216, K=3072: 128-wide 45.7, 192-wide 42.6, 256-wide 47.8;
// M=80, N=3072, K=12288: 31.1, 41.5, 53.0; M=768, N=9216, K=3072: 65.4, 59.2, 52.3. Two problems pay more for workgroups that share a tile, as twice
// the weights arrive from memory meanwhile (pair_*). us, 128 / 192 / 256 wide at their best / the tile kernel: 195 + 256 rows, N=3072, K=3072 25.9 / 25.1 / 29.1 / 24.7;
// 300 + 300 29.0 / 28.5 / 30.1 / 27.4; 768 + 128 35.2 / 34.8 / 35.6 / 30.4; N=9216: 128 + 40 37.3 / 37.4 / 38.2 / 35.8, 256 + 64 39.8 / 44.2 / 44.6 / 39.4. Choosing among
// these forms and the tile kernel by the two plans' times takes 0.63 % longer than the best of all over 110 pairs of 2 to 8 row tiles, 0.02 % over 60 of 9 to 20;
// with one problem's times for two 2.4 and 0.1 %, with what is paid added behind the choice of the form 0.83 %.
struct StreamkPlan { int bm, bn, mt0, m_tiles, groups; float us; };

static StreamkPlan plan_streamk(int M0, int M1, int N, int K, int cus) {
  StreamkPlan best{};
  const int most = cus < kGemmMaxWorkers ? cus : kGemmMaxWorkers;
  StreamkPlan p;
  p.bm = M0 <= 64 && M1 <= 64 ? 64 : kGemmBM;  // 64-row tiles where no problem has more rows than that
  p.mt0 = row_tiles(M0, p.bm);
  p.m_tiles = p.mt0 + (M1 > 0 ? row_tiles(M1, p.bm) : 0);
  if (p.m_tiles > most) return best;
  const int k_steps = K / kGemmBK, room = most / p.m_tiles;
  // pair_*: what two problems pay beyond that, as twice the weights arrive from memory meanwhile
  static const struct { int bn; float step, share, range, pair_share, pair_range; } kinds[3] = {
      {128, .62f, 1.2f, 4.f, 0.f, 2.f}, {192, .74f, 2.f, 10.f, 3.f, 0.f}, {256, .88f, 2.7f, 16.f, 5.3f, 0.f}};
  for (const auto& k : kinds) {
    const float share = k.share + (M1 > 0 ? k.pair_share : 0.f), range = k.range + (M1 > 0 ? k.pair_range : 0.f);
    if (p.bm == 64 && k.bn != 128) continue;
    const int n_tiles = (N + k.bn - 1) / k.bn;
    if (static_cast<int64_t>(p.m_tiles) * n_tiles * 8 > static_cast<int64_t>(kGemmCounterBytes)) continue;
    p.bn = k.bn;
    auto offer = [&](int groups, float us) {
      p.groups = groups;
      p.us = us;
      if (best.groups == 0 || us < best.us) best = p;
    };
    if (room >= n_tiles) {
      const int split = room / n_tiles < k_steps ? room / n_tiles : k_steps;
      offer(n_tiles * split, 8.f + (k_steps + split - 1) / split * k.step + (split - 1) * share);
    }
    const int64_t total = static_cast<int64_t>(n_tiles) * k_steps;
    const int groups = total < room ? static_cast<int>(total) : room;
    const int64_t steps = (total + groups - 1) / groups;
    offer(groups, 8.f + steps * k.step + range + static_cast<float>(steps / k_steps) * 6.f);
  }
  return best;
}

float gemm_streamk_us(int M0, int M1, int N, int K, int cus) {
  const StreamkPlan p = plan_streamk(M0, M1, N, K, cus);
  return p.groups > 0 ? p.us : 0.f;
}

int launch_gemm_streamk(const GemmCall* c, int count, int dtype, void* scratch, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const StreamkPlan plan = plan_streamk(c[0].M, count > 1 ? c[1].M : 0, c[0].N, c[0].K, cus);
  if (plan.groups == 0) { set_error("odit_linear: too many output tiles for the stream-K kernel"); return ODIT_ENOTSUP; }
  GemmParams p;
  p.p0 = problem_of(c[0]);
  p.p1 = count > 1 ? problem_of(c[1]) : p.p0;
  p.N = c[0].N;
  p.k_steps = c[0].K / kGemmBK;
  p.mt0 = plan.mt0;
  p.m_tiles = plan.m_tiles;
  const int bm = plan.bm, bn = plan.bn;
  p.total_steps = static_cast<unsigned>((p.N + bn - 1) / bn) * p.k_steps;
  p.groups = plan.groups;
  p.workers = p.groups * p.m_tiles;
  p.counters = static_cast<unsigned long long*>(scratch);
  p.epoch = next_ticket_epoch();
  p.slots = static_cast<char*>(scratch) + kGemmCounterBytes;
  const dim3 grid(p.workers), block(kWaves * 64);
#define ODIT_STREAMK(T)                                                                                        \
  do {                                                                                                         \
    if (bm == 64) hipLaunchKernelGGL((gemm_streamk_kernel<T, 64, 128>), grid, block, 0, stream, p);              \
    else if (bn == 128) hipLaunchKernelGGL((gemm_streamk_kernel<T, 128, 128>), grid, block, 0, stream, p);       \
    else if (bn == 192) hipLaunchKernelGGL((gemm_streamk_kernel<T, 128, 192>), grid, block, 0, stream, p);       \
    else hipLaunchKernelGGL((gemm_streamk_kernel<T, 128, 256>), grid, block, 0, stream, p);                      \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_STREAMK(bf16_t);
  else ODIT_STREAMK(f16_t);
#undef ODIT_STREAMK
  return check_launch("odit_linear (stream-K kernel)");
}

}  // namespace odit
