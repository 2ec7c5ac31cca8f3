// K1, production variant: software-pipelined flash attention whose K/V tiles go from global memory
// straight into LDS (buffer_load ... lds), with no staging registers, no LDS store instructions and
// no per-tile address arithmetic.
//
// Tile movement. A tile is 64 keys x D elements, row-major, unpadded (256 B rows for D = 128). One
// `buffer_load_dwordx4 ... lds` of a wavefront fills 1 KB of LDS: lane l's 16 bytes land at
// base + 16*l (measured), so the PLACE is fixed and the lane picks WHAT it fetches. Lane l therefore
// fetches, for tile row r = 4*i + l/16 and physical 16-byte chunk pc = l%16, the logical chunk
// pc ^ f(r): the swizzle lives in the global address. Per-lane byte offsets are computed once; the
// tile index only moves a scalar offset. The buffer descriptor's size is the end of the last valid
// key row, so rows past Sk read as zeros without any clamping.
//   K:  f(r) = r % 16       a quarter-wave (16 key rows, one chunk column) of a ds_read_b128 covers
//                           all 64 banks
//   V:  f(r) = 4 * (r % 4)  the 4 keys x 4 eight-byte words of two ds_read_b64_tr_b16 groups cover
//                           all 64 banks
// Fragment addresses then are (per-lane base) XOR (a compile-time constant) plus an immediate.
//
// Vector work. The softmax's vector instructions bound the launches beside the part's power, so a tile has only those that it cannot do
// without (32 exp2, 32 multiply-adds, 32 adds, 16 packs, 16 maxima): the row maximum is formed over the lane halves only where a lane
// sees the running one left behind, its exponent is kept from there (settle_max), the next scores' maximum is formed an
// instruction or two behind each MFMA of stage B instead of in one piece behind the second, and there is one path of selects for
// excluded keys (mask_and_max). us, before / now, the same bits:
//   D=128  B=1 S=16384 H=40  4645 / 4572 (on zeros, without the power limit, 3548 / 3430)    B=2 S=4352 H=24  439 / 432
//          B=1 S=4608 H=24  248 / 243      B=1 S=1536 H=24  42.7 / 41.2
//   D=64 (with fills_two's rule)  B=2 S=4178 H=4  67.6 / 64.0     B=1 S=4096 H=8  55.6 / 51.2     B=1 S=8192 H=16  298 / 293
//          B=2 S=4352 H=24  276 / 260     B=2 S=1357 H=32 f16 with a mask 53.8 / 42.4, padded row 42.0 / 34.2
// v_mfma_f32_16x16x32 (two groups of 16 queries a wavefront) draws less power for the same products (a loop of nothing else: 2054
// TFLOP/s on random operands, 32x32x16 1784; on zeros 2415 and 2440) and is twice as many instructions to issue. It took the first
// launch to 4424 and zeros to 3869, but a video step of 32760 keys, whose probabilities are nearly even, to 0.997 of the time before
// where this form takes it to 0.99, and wavefronts alone on their SIMD 8 % longer (B=2 S=4178 H=4 73.0): not kept. Sums of the
// probabilities in stage B, packing pinned in stage A, the first V fragments ahead of the stages' barrier, other priorities and
// more fragments ahead: all slower.
//
// Everything else (transposed S^T = K Q^T / O^T = V^T P^T formulation, one query per lane, lazy
// rescale, stage A = next-tile QK^T MFMAs interleaved with this tile's exp2 work, stage B = PV, one
// barrier per tile - two in the anti-phase form of 8 wavefronts, see NW below -, XCD-aware workgroup order)
// is as in attn_fwd_pipe_kernel.
//
// Key mask. Before the first scores each wavefront turns its share of the mask row into one 64-bit word per key tile (a
// ballot over the tile's 64 bytes; keys past Sk are zero bits) in LDS. A tile whose word is all ones then runs like a tile of
// a launch without a mask, any other one selects its scores by the word's bits, wave-uniform both. Read as bytes from
// global memory at every tile, 32 loads, clamps and selects per lane, a mask cost 34 to 88 % whatever was in it. us, bf16,
// no mask / all-true mask, bytes / all-true mask, words:
//   B=2 S=4352 H=24 D=128  439 / 737 / 451      B=1 S=4608 H=24 D=128  249 / 469 / 258
//   B=2 S=592 H=24 D=128   18.4 / 26.8 / 18.8   B=2 S=4352 H=24 D=64   279 / 505 / 289
// (and 490 / 290 / 20.6 / 333 with a random mask, where every tile is mixed; at D=64 now 260 / - / 272).
// Past kMaskWords tiles, and in the persistent form, whose units change the batch row, the word is formed at each tile, from one byte a lane.
// With the words a unit ends with the last tile that has a live key: the tiles behind it would add zero probabilities (and are not
// read: a NaN among their values does not reach the rows). Together with spread_batch below, one batch row padded to 40 % of
// the other's keys, us, f16, before / now, and the same with an all-true mask (what a launch gains depends on the padding: with
// three drawn lengths of the second row the first shape takes 46 to 53):
//   B=2 S=1357 H=32 (8 of keys) D=64  60.1 / 43.0, 56.0 / 56.2    B=2 S=1195 H=24 D=128  45.8 / 36.4, 46.1 / 45.4
//   B=2 S=4352 H=24 D=64              320 / 296, 298 / 299        B=2 S=4352 H=24 D=128  485 / 468, 473 / 474
// (at D=64 since then, three workgroups to a compute unit: 34, 42 and 270, 272)
// Passing over the dead tiles between live ones too, by a list of the live ones, cost 1 to 2 % of every masked launch in the tile
// loop, and skipping those ahead of the first live one 0.3 us of a second copy of the first scores.
//
// Persistent form (MODE 2), a measurement aid that no default launch uses (ODIT_ATTN_PERSISTENT=1 in the
// environment turns it on for launches of 4-wavefront workgroups, i.e. with ODIT_ATTN_WAVES=4 at head size 128). With
// more units than workgroup slots the launch has as many workgroups as run at once, and each runs unit after unit as ONE stream of key tiles: the tile pipeline runs across the unit
// boundary. Units are handed out dynamically: every XCD owns a contiguous eighth of the units (neighbours in
// (q block, head) order share keys and values in its L2), its workgroups start on the first ones and draw the
// next from the XCD's ticket word in scratch whenever they begin a unit, one unit ahead of need, so the draw's
// latency hides behind that unit's first tile. While a unit's last tiles are multiplied, the K and V tiles of
// the next unit's first keys are already on their way into LDS; the last tile's stage A computes the next
// unit's first scores from that unit's queries (fetched a tile earlier into the fragment registers the finished
// unit no longer needs); after the last tile's stage B the finished unit is normalised and stored and the
// running maximum, sum and accumulators start again. A unit then costs its key tiles and one fetch of its
// queries, not a workgroup dispatch, a cold prologue and a drained pipeline at its end.
// What it measured (bf16, D = 128, us, one workgroup per unit / persistent, same process, same box):
//   B=2 S=4352 H=24 (3.19 rounds)  506 / 532      B=2 S=4096 H=24 (3.00 rounds)  433 / 447
//   B=1 S=4608 H=24 (1.69 rounds)  306 / 316      B=2 S=32760 H=40 (40 rounds)   39709 / 41187
// i.e. 3 to 5 % slower everywhere, also at 40 units per workgroup where the boundaries no longer matter: the
// steady-state tile loop itself is slower. It carries the next unit's state and the boundary's branches in 97 of
// 102 scalar registers, so the tile loads' LDS destinations and the fragment addresses are formed again in every
// tile instead of being held: the hardware counters show 5.07 vector instructions per MFMA against 4.54 and the
// matrix pipe busy 54.0 % of the cycles against 60.1 %. And what it saves is little: at 8 key tiles per unit, where
// a unit's fixed cost (8 us: dispatch, cold first tiles, first scores, store) is a third of the unit, it runs in
// the time of one workgroup per unit (899 / 901 us at 32760 queries x 512 keys x 40 heads), so its boundary costs
// what a dispatch and a cold start cost. With a fixed assignment of units (w, w + W, ...) instead of the ticket
// words it was 6 % slower: compute units do not all run at one speed, and the dispatcher (or the tickets) gives
// the faster ones more work. Neither form removes the cost of a last round that is partly filled: that needs
// units cut along the keys (MODE 1).
#include <stddef.h>

#include <cstdlib>

#include "attn_common.h"
#include "attn_tail.h"

// LDS fragment reads issued ahead of the MFMA that consumes them (K: 16-byte reads, V: pairs of
// transpose reads); overridable for tuning builds.
#ifndef ODIT_ATTN_KPF
#define ODIT_ATTN_KPF 3
#endif
#ifndef ODIT_ATTN_VPF
#define ODIT_ATTN_VPF 3
#endif

namespace odit {

// A kernel argument fetched again from the argument segment at the point of use (a scalar load the compiler can
// neither hoist nor merge with others). The persistent form reads what it needs at a unit boundary this way:
// taken from the by-value argument struct, those fields would be held in scalar registers across the whole tile
// loop, which has none to spare.
template <typename V> __device__ __forceinline__ V kernel_arg(size_t offset) {
  typedef __attribute__((address_space(4))) const char* arg_ptr;
  arg_ptr base = (arg_ptr)__builtin_amdgcn_kernarg_segment_ptr();
  return *(const volatile __attribute__((address_space(4))) V*)(base + offset);
}
#define ODIT_ARG(field) (PERSIST ? kernel_arg<decltype(AttnParams::field)>(offsetof(AttnParams, field)) : p.field)

typedef short s16x4_d __attribute__((ext_vector_type(4)));
typedef short s16x8_d __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4_d* lds_s16x4_p;
typedef __attribute__((address_space(3))) void* lds_void_p;

// MODE 0: workgroup i owns unit i (a q block of one head of one batch row), all keys.
// MODE 1: launched after the full rounds for the units that are left over: workgroup i owns key
//         tiles [jt0, n_tiles) of unit n_full + i / key_chunks and leaves an unnormalised partial
//         result in scratch for attn_merge_kernel.
// MODE 2: persistent, see above.
// MODE 3, 4: 0 and 1 for a key mask held as words. MODE 5: 3 with the batch rows spread over the XCDs (spread_batch).
// MODE 6, 7, 8: 0, 3 and 5 of head size 64 with two workgroups per compute unit in the place of three (fills_two).
// Separate instantiations, so the extra bookkeeping of one cannot disturb the register allocation of another (that of the
// words in the launches without a mask: 452 -> 460 us at B=2 S=4352 H=24 D=128, 252 -> 262 at B=1 S=4608).
constexpr int kMaskWords = 1024;  // 8 KB of LDS: two workgroups of D = 128 still fit a compute unit (144 of 160 KB)

// Wavefronts on a SIMD, which is workgroups of 4 wavefronts on a compute unit: stated, both ways, because at head size 64 the registers
// that a form happens to take (162 to 174, three wavefronts up to 168) would settle it otherwise.
constexpr int kWavesPerSimd(int D, int NW, int MODE) { return D == 64 && NW == 4 && (MODE == 0 || MODE == 3 || MODE == 5) ? 3 : 2; }

template <typename T, int D, int NW, int MODE>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd(D, NW, MODE), kWavesPerSimd(D, NW, MODE))))
void attn_fwd_dma_kernel(const AttnParams p) {
  constexpr bool TAIL = MODE == 1 || MODE == 4;
  constexpr bool PERSIST = MODE == 2;
  constexpr bool WORDS = MODE >= 3 && MODE != 6;
  constexpr bool SPREAD = MODE == 5 || MODE == 8;
  using M = Mma<T>;
  using frag = typename M::frag;
  constexpr int BN = 64;
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int ROWB = D * 2;                 // bytes per tile row
  constexpr int CPR = ROWB / 16;              // 16-byte chunks per row (16 for D=128, 8 for D=64)
  constexpr int RPI = 64 / CPR;               // tile rows filled by one wave instruction (4 or 8)
  constexpr int TILEB = BN * ROWB;            // bytes per tile
  constexpr int NINST = BN / RPI;             // wave instructions per tile (16 or 8)
  // NW = 8 is the anti-phase form: the workgroup's two wavefronts on a SIMD (w and w + 4) run the same tile loop
  // half a tile apart, held there by a second barrier between the stages, so one's stage A (exp2 and the other
  // vector work, with the next scores' MFMAs) always meets the other's stage B (MFMAs and LDS reads only). Wavefronts
  // 0-3 fetch the K tiles, 4-7 the V tiles, each group at the start of its own stage A.
  constexpr bool PP = NW == 8;
  static_assert(!(PP && PERSIST), "the persistent form has no anti-phase variant");
  constexpr int NWL = PP ? 4 : NW;              // wavefronts that fetch one tile
  constexpr int IPW = (NINST + NWL - 1) / NWL;  // ... per wavefront
  static_assert(NINST % NWL == 0, "tile loads must divide evenly over the wavefronts");
  constexpr int BM = NW * 32;

  __shared__ __attribute__((aligned(1024))) char lds[4 * TILEB];  // K0 K1 V0 V1
  char* const Kb = lds;
  char* const Vb = lds + 2 * TILEB;
  constexpr int kKoff = 0, kVoff = 2 * TILEB;  // the same as byte offsets, for the tile loads' LDS destinations

  const int n_tiles_all = (p.Sk + BN - 1) / BN;
  int pid, jt0 = 0, n_tiles = n_tiles_all;
  const int part = blockIdx.x;
  // persistent form: the unit after the current one (-1: none, or not drawn yet)
  int next_pid = -1;
  static_assert(MODE < 6 || (D == 64 && NW == 4), "two workgroups per compute unit in the place of three: head size 64");
  __shared__ int next_unit_box;  // thread 0's draw, handed to the workgroup across a tile's barrier
  __shared__ uint64_t mask_words[WORDS ? kMaskWords : 1];  // of key tiles jt0, jt0 + 1, ...
  if constexpr (!TAIL && !PERSIST) {
    pid = xcd_remap(blockIdx.x, p.n_full);
  } else if constexpr (TAIL) {  // this workgroup covers key tiles [jt0, n_tiles) of unit pid (jt0 is even)
    pid = p.n_full + part / p.key_chunks;
    jt0 = (part % p.key_chunks) * p.tiles_per_chunk;
    n_tiles = jt0 + p.tiles_per_chunk < n_tiles_all ? jt0 + p.tiles_per_chunk : n_tiles_all;
  } else {
    // gridDim.x = W workgroups, a multiple of the XCD count, all resident; hardware puts workgroup w on XCD
    // w % 8. XCD x owns units [x_lo, x_hi); its W / 8 workgroups start on the first W / 8 of them.
    const int xcd = part % kNumXcd;
    const int x_lo = static_cast<int>(static_cast<int64_t>(p.n_full) * xcd / kNumXcd);
    const int x_hi = static_cast<int>(static_cast<int64_t>(p.n_full) * (xcd + 1) / kNumXcd);
    pid = x_lo + part / kNumXcd;
    if (pid >= x_hi) return;  // fewer units than workgroups on this XCD (before any barrier: the whole workgroup leaves)
  }
  const int tid = threadIdx.x, lane = tid & 63;
  // (a scalar only where three workgroups with mask words leave no vector register for it: two went to memory)
  const int wave = WORDS && kWavesPerSimd(D, NW, MODE) == 3 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int wl = PP ? (wave & 3) : wave;     // this wavefront's share of a tile load
  const bool grp1 = PP && wave >= 4;          // second group of the anti-phase form (wave-uniform)

  // ---- the current unit (fixed for MODE 0 and 1, advanced unit by unit in the persistent form) ----
  int h = (pid / p.n_qblocks) % p.H;
  int b = (pid / p.n_qblocks) / p.H;
  int q0 = (pid % p.n_qblocks) * BM + wave * 32;
  if constexpr (SPREAD) {
    h = blockIdx.x % kNumXcd * (p.H / kNumXcd) + blockIdx.y;
    b = blockIdx.z;
    q0 = blockIdx.x / kNumXcd * BM + wave * 32;
  }

  // buffer descriptors end right after the last valid key row: later rows read as zeros
  const uint32_t k_bytes = static_cast<uint32_t>(((p.Sk - 1) * p.ks_s + D) * 2);
  // value rows [0, k_split) come from v, rows [k_split, Sk) from v_tail (k_split is a whole number of
  // tiles and both share the row stride): two descriptors, picked per tile with scalar selects
  const int v_split_tiles = p.v_tail != nullptr ? p.k_split / BN : n_tiles_all;
  const int v_rows = p.v_tail != nullptr ? p.k_split : p.Sk;
  const uint32_t v_bytes = static_cast<uint32_t>(((v_rows - 1) * p.vs_s + D) * 2);
  const uint32_t v2_bytes = p.v_tail != nullptr ? static_cast<uint32_t>(((p.Sk - p.k_split - 1) * p.vs_s + D) * 2) : v_bytes;
  // raw buffer descriptors {base[31:0], base[47:32] (stride 0), bytes, dword3 = 0x00020000}
  auto make_rsrc = [](const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    u32x4_v r;
    r.x = static_cast<uint32_t>(a); r.y = static_cast<uint32_t>(a >> 32) & 0xffffu; r.z = bytes; r.w = 0x00020000u;
    return r;
  };
  // descriptors of the keys / values / second value tensor of (batch b_, head h_)
  auto k_rsrc_of = [&](int b_, int h_) {
    const int hkv_ = h_ / (ODIT_ARG(H) / ODIT_ARG(Hkv));
    return make_rsrc(static_cast<const T*>(ODIT_ARG(k)) + b_ * ODIT_ARG(ks_b) + hkv_ * ODIT_ARG(ks_h), k_bytes);
  };
  auto v_rsrc_of = [&](int b_, int h_) {
    const int hkv_ = h_ / (ODIT_ARG(H) / ODIT_ARG(Hkv));
    return make_rsrc(static_cast<const T*>(ODIT_ARG(v)) + b_ * ODIT_ARG(vs_b) + hkv_ * ODIT_ARG(vs_h), v_bytes);
  };
  auto v2_rsrc_of = [&](int b_, int h_) {
    const int hkv_ = h_ / (ODIT_ARG(H) / ODIT_ARG(Hkv));
    return make_rsrc(static_cast<const T*>(ODIT_ARG(v_tail)) + b_ * ODIT_ARG(vt_b) + hkv_ * ODIT_ARG(vt_h), v2_bytes);
  };
  u32x4_v krsrc = k_rsrc_of(b, h);
  u32x4_v vrsrc = v_rsrc_of(b, h);
  u32x4_v vrsrc2 = p.v_tail != nullptr ? v2_rsrc_of(b, h) : vrsrc;
  const uint8_t* mrow = p.mask ? p.mask + static_cast<int64_t>(b) * p.Sk : nullptr;
  // persistent form: where the next unit is (valid while next_pid >= 0)
  int n_h = 0, n_b = 0;
  // Thread 0 draws the unit after the current one: the XCD's word is raised to this launch's epoch (a no-op but
  // for the XCD's first draw of the launch), then ticket t names unit x_first + t. Every unit that is run draws
  // once, so the draw with the ticket of the XCD's last unit is the launch's last on this word and puts it back
  // to zero (a launch replayed from a HIP graph carries the same epoch).
  auto draw_next = [&]() {
    if (tid == 0) {
      // the XCD's unit range, worked out again here rather than held in scalar registers for the whole unit
      int xcd = part % kNumXcd;
      asm volatile("" : "+s"(xcd));  // (so that the word's address is formed here, not held in vector registers)
      const int per = static_cast<int>(gridDim.x) / kNumXcd;
      const int x_lo = static_cast<int>(static_cast<int64_t>(p.n_full) * xcd / kNumXcd);
      const int x_hi = static_cast<int>(static_cast<int64_t>(p.n_full) * (xcd + 1) / kNumXcd);
      const int x_first = x_lo + per < x_hi ? x_lo + per : x_hi;  // first unit handed out by ticket
      unsigned long long* word = ODIT_ARG(queue) + xcd * 8;
      __hip_atomic_fetch_max(word, ODIT_ARG(epoch) << 24, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned t = static_cast<unsigned>(__hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) & 0xffffffu;
      if (static_cast<int>(t) == x_hi - x_lo - 1) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int cand = x_first + static_cast<int>(t);
      next_unit_box = cand < x_hi ? cand : -1;
    }
  };
  auto take_next = [&]() {  // behind the barrier that follows draw_next
    next_pid = __builtin_amdgcn_readfirstlane(next_unit_box);
    if (next_pid >= 0) {
      const int bh = next_pid / ODIT_ARG(n_qblocks), heads = ODIT_ARG(H);
      n_h = bh % heads;
      n_b = bh / heads;
    }
  };

  // Per-lane global byte offset of the chunk this lane moves with its wave's FIRST instruction of a tile,
  // relative to the tile's first row; instruction i moves the rows RPI * i further down, which is a scalar
  // term (it goes into the load's scalar offset), and its swizzle differs from the first one's by a constant:
  // for K, row % 16 = (row0 % 16) + (RPI * i) % 16 without a carry (row0 % 16 < RPI), so the chunk index is that
  // of instruction 0 XOR ((RPI * i) % 16 % CPR) - for V (4 * (row % 4), RPI a multiple of 4) it is the same. The
  // XOR is done on the byte offset, which needs row strides that are multiples of the row's own 2 D bytes.
  const int r0 = wl * IPW * RPI + lane / CPR, pc0 = lane % CPR;
  const uint32_t kvoff0 = static_cast<uint32_t>(r0 * p.ks_s * 2) + static_cast<uint32_t>(((pc0 ^ (r0 % 16)) % CPR) * 16);
  const uint32_t vvoff0 = static_cast<uint32_t>(r0 * p.vs_s * 2) + static_cast<uint32_t>(((pc0 ^ (4 * (r0 % 4))) % CPR) * 16);
  const uint32_t k_inst_step = static_cast<uint32_t>(RPI * p.ks_s * 2);
  const uint32_t v_inst_step = static_cast<uint32_t>(RPI * p.vs_s * 2);
  const uint32_t k_tile_step = static_cast<uint32_t>(BN * p.ks_s * 2);
  const uint32_t v_tile_step = static_cast<uint32_t>(BN * p.vs_s * 2);

  // The tile loads are written as inline assembly on purpose. Issued through the compiler's builtin they
  // are known to it as pending LDS writes, and it then puts `s_waitcnt vmcnt(0)` in front of the first V
  // fragment read of every tile (it cannot prove that the XOR-swizzled read addresses miss the buffer
  // being filled): the loads issued at the top of a tile, meant to land a whole tile later, were waited
  // for half a tile after issue. Here the ordering is explicit instead: one `s_waitcnt vmcnt(0)` and one
  // barrier at the end of each tile, before any wave reads the buffers those loads filled.
  // `dst_off` is the tile's byte offset inside the kernel's LDS block: a literal at every call
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_p)lds));
  auto dma_tile = [&](const u32x4_v& rsrc, const bool is_k, uint32_t soff, const int dst_off) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t lds0 = lds_base + static_cast<uint32_t>(dst_off) + static_cast<uint32_t>(wl * IPW * 1024);
    // (the empty asm makes the offset opaque here: otherwise the compiler forms the IPW swizzled offsets once,
    // outside the tile loop, and holds them in registers the loop does not have)
    uint32_t voff0 = is_k ? kvoff0 : vvoff0;
    asm volatile("" : "+v"(voff0));
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds0 + i * 1024);
      const uint32_t voff_i = is_k ? (voff0 ^ static_cast<uint32_t>((((RPI * i) % 16) % CPR) * 16)) : voff0;
      const uint32_t soff_i = soff + static_cast<uint32_t>(i) * (is_k ? k_inst_step : v_inst_step);
      load_lds16<true>(m0v, voff_i, rsrc, soff_i);
    }
#endif
  };

  auto dma_v = [&](int jt, const int dst) {
    const bool second = jt >= v_split_tiles;
    dma_tile(second ? vrsrc2 : vrsrc, false, static_cast<uint32_t>(second ? jt - v_split_tiles : jt) * v_tile_step, dst);
  };
  // the same for tiles of the NEXT unit (persistent form): descriptors made on the spot from (n_b, n_h), a few
  // scalar instructions per tile instead of a dozen scalar registers held for the whole unit
  auto dma_k_next = [&](int jt, const int dst) {
    dma_tile(k_rsrc_of(n_b, n_h), true, static_cast<uint32_t>(jt) * k_tile_step, dst);
  };
  auto dma_v_next = [&](int jt, const int dst) {
    const bool second = jt >= v_split_tiles;
    dma_tile(second ? v2_rsrc_of(n_b, n_h) : v_rsrc_of(n_b, n_h), false,
             static_cast<uint32_t>(second ? jt - v_split_tiles : jt) * v_tile_step, dst);
  };

  // ---- Q fragments stay in registers ----
  frag qf[KS];
  // (the persistent form calls these two inside the tile loop: they take the lane's position from the thread
  // index again, so that nothing of theirs is carried through the loop)
  auto lane_again = [&](int& l32_, int& hh_) {
    int t = tid;
    if constexpr (PERSIST) asm volatile("" : "+v"(t));
    l32_ = t & 31;
    hh_ = (t >> 5) & 1;
  };
  auto load_q = [&](int b_, int h_, int q0_) {
    int l32, hh;
    lane_again(l32, hh);
    int row = q0_ + l32;
    const int rows = ODIT_ARG(Sq);
    row = row < rows ? row : rows - 1;
    const T* qp = static_cast<const T*>(ODIT_ARG(q)) + b_ * ODIT_ARG(qs_b) + h_ * ODIT_ARG(qs_h) + row * ODIT_ARG(qs_s) + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4_v*>(qp + ks * 16));
  };
  load_q(b, h, q0);

  f32x16_v o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f, mc = 0.f;  // mc: m_run as an exponent, 0 before the first score

  const float c = p.scale_log2, c_rescale = fmaxf(c, 0.f);

  // K fragment (kt, ks): row kt*32 + l32, logical chunk 2*ks + hh  ->  chunk (2*ks) ^ (hh ^ l32 % 16)
  const int k_lane = l32 * ROWB + ((((hh ^ (l32 % 16)) % CPR)) << 4);
  // V transpose read, 16-lane group g = lane/16 (d half dh = g&1, key half = hh), lane s = lane%16:
  // key 4*hh + s/4 (+ tile offsets), logical chunk 4*dt + 2*dh + (s%4)/2, 8-byte half (s%4)%2,
  // physical chunk = logical ^ 4*(s/4)  ->  XOR of the dt field only
  const int sq = (lane & 15) >> 2;
  const int dh = (lane >> 4) & 1;
  const int v_lane = (4 * hh + sq) * ROWB + ((((4 * sq) % CPR) ^ (2 * dh + ((lane & 3) >> 1))) << 4) + ((lane & 1) << 3);

  auto qk_plain = [&](const char* kt_base, f32x16_v(&s)[2]) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[kt][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const frag a = __builtin_bit_cast(
            frag, *reinterpret_cast<const u32x4_v*>(kt_base + kt * 32 * ROWB + (k_lane ^ (ks * 32))));
        s[kt] = M::run(a, qf[ks], s[kt]);
      }
  };

  // The lane's maximum of its 32 scores, in 16 instructions (v_maximum3_f32; fmaxf would first put a maximum with itself, which quiets
  // a NaN, in front of every score). A NaN score takes the lane's maximum, which then is not looked at: the query's result is NaN
  // anyway. Not inline assembly, although the scores are matrix results: the vector unit may read those some wait states later
  // only, and it is the compiler that sees to them.
  constexpr int NMAX = 16;
  auto max_step = [&](const f32x16_v(&s)[2], float mx, int n) __attribute__((always_inline)) -> float {
    auto e = [&](int i) __attribute__((always_inline)) { return s[i >> 4][i & 15]; };
    if (n == 0) return __builtin_elementwise_maximum(__builtin_elementwise_maximum(e(0), e(1)), e(2));
    if (n == NMAX - 1) return __builtin_elementwise_maximum(mx, e(31));
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, e(2 * n + 1)), e(2 * n + 2));
  };

  // excluded scores of tile j become -inf (branch-free selects: every lane rewrites all its scores); returns the lane's maximum.
  // w: the tile's mask word (WORDS; formed here otherwise: one path of selects for what is excluded by a mask and by the sequence's
  // end, as with two of them the tiles without either paid 16 to 32 register copies each, 4 % of a launch)
  auto mask_and_max = [&](int j, const uint8_t* mrow, uint64_t w, f32x16_v(&s)[2]) -> float {
    if constexpr (!WORDS) {
      const int keys = p.Sk - j * BN;  // from here to the end (one at least)
      w = keys < BN ? (1ull << keys) - 1 : ~0ull;
      if (mrow != nullptr) w &= __ballot(mrow[lane < keys ? j * BN + lane : p.Sk - 1] != 0);
    }
    // (this lane's keys are 8 g + 4 hh + t of each half of the tile)
    const uint32_t half[2] = {static_cast<uint32_t>(w) >> (4 * hh), static_cast<uint32_t>(w >> 32) >> (4 * hh)};
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float x = s[kt][g * 4 + t];
          s[kt][g * 4 + t] = (half[kt] & (1u << (g * 8 + t))) ? x : -INFINITY;
        }
    float mx = 0.f;
#pragma unroll
    for (int n = 0; n < NMAX; ++n) mx = max_step(s, mx, n);
    return mx;
  };

  // x of the lane 32 further or before
  auto swapped = [&](float x) __attribute__((always_inline)) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(hh ? r[0] : r[1]);
  };
  // mx: the lane's maximum. The row's, over both lane halves, is formed only where the running one is left behind by a factor of 2^8.
  auto settle_max = [&](float mx) __attribute__((always_inline)) {
    if (__any((mx - m_run) * c_rescale > 8.f)) {
      const float m_new = fmaxf(m_run, fmaxf(mx, swapped(mx)));
      const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_safe) * c);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
      m_run = m_new;
      mc = m_safe * c;
    }
  };

  // normalises and stores the finished unit (b, h, q0): the tail of MODE 0 and of every unit of the persistent form
  auto finish_unit = [&]() {
    int l32, hh;
    lane_again(l32, hh);
    const float l_tot = l_run + swapped(l_run);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const int row = q0 + l32;
    if (row < ODIT_ARG(Sq)) {
      // head of the joint sequence in `o`, tail in `o_tail` (out_row_ptr, with the arguments fetched here)
      T* op;
      void* const o_tail = ODIT_ARG(o_tail);
      const int q_split = ODIT_ARG(q_split);
      if (o_tail != nullptr && row >= q_split) {
        op = static_cast<T*>(o_tail) + b * ODIT_ARG(ts_b) + h * ODIT_ARG(ts_h) + static_cast<int64_t>(row - q_split) * ODIT_ARG(ts_s);
      } else {
        op = static_cast<T*>(ODIT_ARG(o)) + b * ODIT_ARG(os_b) + h * ODIT_ARG(os_h) + static_cast<int64_t>(row) * ODIT_ARG(os_s);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
          // A lane has 4 features of every 8, the lane 32 further the others of its row: exchanged, each has 8 in a row and stores 16 bytes, half
          // as many stores as without. us, bf16, 8 bytes a store / 16, the same bits: D = 128 B=2 S=296 H=24 12.4 / 11.4, B=2 S=1195 44.3 / 42.6,
          // 32760 queries x 512 keys H=40 433 / 403, B=2 S=4352 H=24 418 / 411; D = 64 9.0 / 8.5, 29.4 / 28.7, 237 / 225, 257 / 255. Whole rows,
          // turned round in the tiles' LDS first: 12.5, 42.9, 412, 415; 9.2, 29.6, 236, 256.
          auto pair = [&](int e) __attribute__((always_inline)) {
            return __builtin_amdgcn_permlane32_swap(M::pack2(o[dt][g * 4 + e] * inv, o[dt][g * 4 + e + 1] * inv),
                                                    M::pack2(o[dt][g * 4 + e + 4] * inv, o[dt][g * 4 + e + 5] * inv), false, false);
          };
          const auto lo = pair(0), hi = pair(2);
          u32x4_v w;
          w.x = lo[0]; w.y = hi[0]; w.z = lo[1]; w.w = hi[1];
          *reinterpret_cast<u32x4_v*>(op + dt * 32 + g * 8 + hh * 8) = w;
          // (in the persistent form this runs inside the tile loop, with the next unit's queries and first scores
          // live: the values go out one store at a time instead of being formed all at once)
          if constexpr (PERSIST) __builtin_amdgcn_sched_barrier(0);
        }
      float* const lse_out = ODIT_ARG(lse);
      if (lse_out != nullptr && hh == 0) {
        const float lse = l_tot > 0.f ? m_run * ODIT_ARG(scale) + __logf(l_tot) : -INFINITY;
        lse_out[(static_cast<int64_t>(b) * ODIT_ARG(H) + h) * ODIT_ARG(Sq) + row] = lse;
      }
    }
  };

  // Tile j of the current unit. In the persistent form the tile after a unit's last one is tile 0 of the
  // workgroup's next unit (`cross`), and the tile after that its tile 1.
  // `buf` (the LDS buffer pair of this tile: the parity of its running index) is a literal at every call, so the
  // LDS addresses below are compile-time offsets.
  auto tile = [&](int j, const int buf, f32x16_v(&s_cur)[2], f32x16_v(&s_next)[2]) {
    const bool last = j + 1 == n_tiles;
    const bool cross = PERSIST && last && next_pid >= 0;
    const bool has_next = !last || cross;
    // buffers K[buf] (held K(j), consumed last tile) and V[buf^1] (held V(j-1)) are free now
    // (anti-phase form: the first group fetches K, the second V; K(j) was last read by the second group's stage A
    // of tile j - 1, half a tile before the first group gets here, V(j-1) by the second group's own stage B)
    if (!PP || !grp1) {
      if (j + 2 < n_tiles) {
        dma_tile(krsrc, true, static_cast<uint32_t>(j + 2) * k_tile_step, kKoff + buf * TILEB);
      } else if (PERSIST && next_pid >= 0) {
        dma_k_next(j + 2 - n_tiles, kKoff + buf * TILEB);
      }
    }
    if constexpr (PERSIST) {
      if (j == 0) draw_next();  // the answer is in the box when this tile's barrier has been passed
    }
    if (!PP || grp1) {
      if (!last) {
        dma_v(j + 1, kVoff + (buf ^ 1) * TILEB);
      } else if (cross) {
        dma_v_next(0, kVoff + (buf ^ 1) * TILEB);
      }
    }
    // the tile whose scores stage A computes, and the mask row of its unit
    const int jn = last ? 0 : j + 1;
    const uint8_t* mrow_n = cross ? (p.mask ? p.mask + static_cast<int64_t>(n_b) * p.Sk : nullptr) : mrow;  // (p.mask and p.Sk are live in the tile loop anyway)

    // (Row sums in fp32 from the unrounded probabilities. Summing the packed pairs with v_dot2c_f32_bf16, one
    // instruction per pair instead of two adds, measured 4 % slower at D = 128, with one chain or four.)
    uint32_t pf[2][2][4];
    float psum = 0.f;
    // Stage A mixes this wave's MFMAs with its exp2 work; giving it issue priority over the SIMD's other
    // wave (which is then mostly in its MFMA + LDS-read stage B) measured +5 % at 32760 keys, +9 % at
    // batch 1 / 4608 keys and nothing lost at the 4352-token, batch-2 shape.
    __builtin_amdgcn_s_setprio(2);
    // ---- stage A ----
    if (has_next) {
      const char* kt_base = Kb + (buf ^ 1) * TILEB;
      // (opaque copy: the KS swizzled variants of the lane offset are formed again in every tile, one XOR each,
      // instead of being carried through the loop in KS registers)
      int k_lane_t = k_lane;
      if constexpr (PERSIST) asm volatile("" : "+v"(k_lane_t));
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e) s_next[kt][e] = 0.f;
      constexpr int KPF = ODIT_ATTN_KPF;  // K fragments in flight ahead of the MFMA that consumes them
      u32x4_v kfr[KPF + 1];
      auto k_fetch = [&](int i) {
        const int ks = i >> 1, kt = i & 1;
        kfr[i % (KPF + 1)] = *reinterpret_cast<const u32x4_v*>(kt_base + kt * 32 * ROWB + (k_lane_t ^ (ks * 32)));
      };
#pragma unroll
      for (int i = 0; i < KPF; ++i) k_fetch(i);
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        if (i + KPF < 2 * KS) k_fetch(i + KPF);
        const int ks = i >> 1, kt = i & 1;
        s_next[kt] = M::run(__builtin_bit_cast(frag, kfr[i % (KPF + 1)]), qf[ks], s_next[kt]);
        constexpr int PAIRS = 16 / (2 * KS) > 0 ? 16 / (2 * KS) : 1;
#pragma unroll
        for (int q = 0; q < PAIRS; ++q) {
          const int pi = i * PAIRS + q;
          if (pi < 16) {
            const int pkt = pi >> 3, e0 = (pi & 7) * 2;
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s_cur[pkt][e0], c, -mc));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(s_cur[pkt][e0 + 1], c, -mc));
            psum += p0 + p1;
            pf[pkt][(pi & 7) >> 2][pi & 3] = M::pack2(p0, p1);
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // pin: fetch(i+KPF), MFMA(i), this step's exp2 work
      }
    } else {
      // (an opaque copy of the offset: were the two branches' exponent arguments the same expressions, the
      // compiler would form all 32 ahead of the branch, out of the MFMAs' shadow and in 32 more registers)
      float mc_t = mc;
      asm volatile("" : "+v"(mc_t));
#pragma unroll
      for (int pi = 0; pi < 16; ++pi) {
        const int pkt = pi >> 3, e0 = (pi & 7) * 2;
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s_cur[pkt][e0], c, -mc_t));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s_cur[pkt][e0 + 1], c, -mc_t));
        psum += p0 + p1;
        pf[pkt][(pi & 7) >> 2][pi & 3] = M::pack2(p0, p1);
      }
    }
    l_run += psum;
    if constexpr (PERSIST) {
      // The next unit's queries replace this unit's once its last scores have been formed, a tile before they are
      // used: they land behind this tile's closing wait. (Loaded at the top of the tile that uses them, the
      // compiler's own wait for them, which it has to place on every trip through the loop, also waits for the
      // tile loads it does not know of.)
      if (j + 2 == n_tiles && next_pid >= 0)
        load_q(n_b, n_h, (next_pid - (n_b * ODIT_ARG(H) + n_h) * ODIT_ARG(n_qblocks)) * BM + wave * 32);
    }

    __builtin_amdgcn_s_setprio(0);
    if constexpr (PP) {
      // the stages' boundary: the two groups swap roles here. A bare barrier: no wavefront writes LDS, and the tile
      // loads in flight are waited for at the end of the tile, not here.
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- stage B: O^T += V(j)^T P(j)^T ----
    // 4*DT steps, head-dim tile innermost so that consecutive MFMAs hit different accumulators and one
    // P fragment serves DT of them; the two transpose reads of step n + PF are issued before the MFMA
    // of step n, so LDS latency is covered by PF matrix instructions. The in-lane row maximum of
    // S(j+1) — vector work with nothing to wait for — is placed in the shadow of these MFMAs.
    const char* vt_base = Vb + buf * TILEB;
    int v_lane_t = v_lane;  // (opaque copy, as for the key fragments)
    if constexpr (PERSIST) asm volatile("" : "+v"(v_lane_t));
    constexpr int NSTEP = 4 * DT;
    constexpr int PF = ODIT_ATTN_VPF;
    s16x4_d vlo[PF + 1], vhi[PF + 1];
    auto v_fetch = [&](int step) {
      const int dt = step % DT, kt = (step / DT) >> 1, g2 = (step / DT) & 1;
      const char* vp = vt_base + (kt * 32 + g2 * 16) * ROWB + (v_lane_t ^ ((dt * 64) % ROWB));
      vlo[step % (PF + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_p)(vp));
      vhi[step % (PF + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_p)(vp + 8 * ROWB));
    };
    bool plain_next = has_next && mrow_n == nullptr && (jn + 1) * BN <= p.Sk;  // no exclusions in the next scores
    uint64_t word = 0;  // (the same in every lane)
    if constexpr (WORDS) {
      if (has_next) word = mask_words[jn - jt0];
    }
    float mx = 0.f;
#pragma unroll
    for (int st = 0; st < PF; ++st) v_fetch(st);
#pragma unroll
    for (int st = 0; st < NSTEP; ++st) {
      if (st + PF < NSTEP) v_fetch(st + PF);
      const int dt = st % DT, kt = (st / DT) >> 1, g2 = (st / DT) & 1;
      const s16x8_d av = __builtin_shufflevector(vlo[st % (PF + 1)], vhi[st % (PF + 1)], 0, 1, 2, 3, 4, 5, 6, 7);
      u32x4_v pb;
      pb.x = pf[kt][g2][0]; pb.y = pf[kt][g2][1]; pb.z = pf[kt][g2][2]; pb.w = pf[kt][g2][3];
      o[dt] = M::run(__builtin_bit_cast(frag, av), __builtin_bit_cast(frag, pb), o[dt]);
      if constexpr (WORDS) {
        if (st == 1) {
          const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(word));
          const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(word >> 32));
          plain_next = has_next && (lo & hi) == ~0u;
        }
      }
      // (the next scores' maximum, an instruction or two behind each MFMA, where the empty asm holds it: it would sink below the test of
      // plain_next otherwise, 264 units of head size 64 65 -> 68 us; formed again where keys are excluded)
      constexpr int EACH = (NMAX + NSTEP - 2) / (NSTEP - 1);
      if (st > 0) {
#pragma unroll
        for (int n = (st - 1) * EACH; n < st * EACH && n < NMAX; ++n) mx = max_step(s_next, mx, n);
        asm volatile("" : "+v"(mx));
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the reads of step st+PF ahead of this MFMA
    }
    if (has_next && !plain_next) {
      mx = mask_and_max(jn, mrow_n, word, s_next);
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's tile loads have landed in LDS
    __syncthreads();
    if constexpr (PERSIST) {
      if (j == 0) take_next();
      if (last) {
        finish_unit();
        if (cross) {  // the next unit becomes the current one; its running maximum, sum and accumulators start over
          h = n_h; b = n_b;
          q0 = (next_pid - (n_b * ODIT_ARG(H) + n_h) * ODIT_ARG(n_qblocks)) * BM + wave * 32;
          krsrc = k_rsrc_of(b, h);
          vrsrc = v_rsrc_of(b, h);
          vrsrc2 = p.v_tail != nullptr ? v2_rsrc_of(b, h) : vrsrc;
          mrow = mrow_n;
          pid = next_pid;
          next_pid = -1;  // drawn during the new unit's first tile
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
          m_run = -INFINITY;
          l_run = mc = 0.f;
        }
      }
    }
    if (has_next) settle_max(mx);
  };

  // ---- prologue (jt0 is even, so tile j always lives in buffer j & 1) ----
  if (!PP || !grp1) dma_tile(krsrc, true, static_cast<uint32_t>(jt0) * k_tile_step, kKoff);
  if (!PP || grp1) dma_v(jt0, kVoff);
  if ((!PP || !grp1) && jt0 + 1 < n_tiles) dma_tile(krsrc, true, static_cast<uint32_t>(jt0 + 1) * k_tile_step, kKoff + TILEB);
  if constexpr (WORDS) {  // behind the first tile loads; up to MB independent loads per memory round trip
    constexpr int MB = 8;
    for (int j0 = jt0 + __builtin_amdgcn_readfirstlane(wave); j0 < n_tiles; j0 += MB * NW) {
      uint8_t m[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int key = (j0 + i * NW) * BN + lane;
        if (j0 + i * NW < n_tiles) m[i] = mrow[key < p.Sk ? key : p.Sk - 1];
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int j = j0 + i * NW;
        if (j < n_tiles) {  // (wave-uniform)
          const uint64_t w = __ballot((j * BN + lane < p.Sk) & (m[i] != 0));
          if (lane == 0) mask_words[j - jt0] = w;
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  f32x16_v sa[2], sb[2];
  uint64_t w = 0;
  if constexpr (WORDS) w = jt0 + lane < n_tiles ? mask_words[lane] : 0;
  qk_plain(Kb, sa);
  {
    uint64_t word = 0;
    if constexpr (WORDS) word = mask_words[0];
    settle_max(mask_and_max(jt0, mrow, word, sa));
  }
  if (WORDS && n_tiles - jt0 > 1) {
    // the unit ends with its last tile that has a live key (the same in every wavefront); where none has, with the first
    int end = jt0 + 1;
    for (int base = jt0;;) {
      const uint64_t live = __ballot(w != 0);
      if (live != 0) end = base + 64 - __builtin_clzll(live);
      base += 64;
      if (base >= n_tiles) break;
      w = base + lane < n_tiles ? mask_words[base + lane - jt0] : 0;
    }
    n_tiles = end;
  }
  // every wavefront has read the first K tile: the loop's first tile load overwrites it
  __syncthreads();
  if constexpr (PP) {
    // the second group enters the loop one barrier, i.e. half a tile, behind the first (which makes up for it
    // behind the loop)
    if (grp1) asm volatile("s_barrier" ::: "memory");
  }

  if constexpr (PERSIST) {
    // one stream of tiles over all units this workgroup gets; every unit stores itself behind its last tile, and
    // the stream ends behind a unit that found the XCD's range exhausted (every wave sees the same next_pid)
    int j = 0;
    for (;;) {  // a tile's buffer pair is the parity of its index in this stream
      bool done = j + 1 == n_tiles && next_pid < 0;
      tile(j, 0, sa, sb);
      if (done) break;
      j = j + 1 == n_tiles ? 0 : j + 1;
      done = j + 1 == n_tiles && next_pid < 0;
      tile(j, 1, sb, sa);
      if (done) break;
      j = j + 1 == n_tiles ? 0 : j + 1;
    }
    return;
  } else {
    for (int j = jt0; j < n_tiles; j += 2) {  // jt0 is even
      tile(j, 0, sa, sb);
      if (j + 1 < n_tiles) tile(j + 1, 1, sb, sa);
    }
    if constexpr (PP) {
      if (!grp1) asm volatile("s_barrier" ::: "memory");
    }
  }

  // ---- epilogue ----
  if constexpr (TAIL) {
    const float l_tot = l_run + swapped(l_run);
    // partial result of a key range: unnormalised O (fp32, [BM][D] per part) and the row's (m, l)
    float* wo = p.ws + (static_cast<int64_t>(part) * BM + wave * 32 + l32) * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4_v w4;
        w4.x = o[dt][g * 4 + 0]; w4.y = o[dt][g * 4 + 1]; w4.z = o[dt][g * 4 + 2]; w4.w = o[dt][g * 4 + 3];
        *reinterpret_cast<f32x4_v*>(wo + dt * 32 + g * 8 + hh * 4) = w4;
      }
    if (hh == 0) {
      float* ml = p.ws + static_cast<int64_t>(gridDim.x) * BM * D +
                  (static_cast<int64_t>(part) * BM + wave * 32 + l32) * 2;
      ml[0] = m_run;
      ml[1] = l_tot;
    }
    return;
  }
  finish_unit();
}

// The persistent form is a measurement aid, off unless the environment says ODIT_ATTN_PERSISTENT=1 when the
// library makes its first attention launch: with it every shape measured ran 3 to 6 % slower than one workgroup
// per unit (its tile loop is slower than what it saves at the unit boundaries, see the header comment).
#ifndef ODIT_ATTN_PERSISTENT_DEFAULT
#define ODIT_ATTN_PERSISTENT_DEFAULT 0
#endif
static bool persistent_form_on() {
  static const bool on = [] {
    const char* e = getenv("ODIT_ATTN_PERSISTENT");
    return e != nullptr ? e[0] == '1' : ODIT_ATTN_PERSISTENT_DEFAULT != 0;
  }();
  return on;
}

// Workgroups of the persistent form for `units` whole units of `n_tiles` key tiles each on `slots` workgroup
// slots, or 0 when every unit gets a workgroup of its own (no more units than slots, or units too short for the
// next unit to be known before its first tiles are fetched).
static int persistent_workgroups(int units, int n_tiles, int slots, int nw) {
  const int W = slots - slots % kNumXcd;
  if (!persistent_form_on() || nw != 4 || W < kNumXcd || units <= W || n_tiles < 4 || units >= (1 << 26)) return 0;  // tickets have 24 bits
  return W;
}

// Batch rows of a masked launch differ in their live tiles, and xcd_remap gives whole batch rows to some of the XCDs: those with
// the longest row finish last (B=2, one row of 22 tiles and one of 9, 704 units: the XCDs 0 to 3 had 88 units of 22 tiles each).
// Where the heads divide evenly every XCD gets its share of each row's heads instead, as many in all (keys and values are shared
// in its L2 as before), by a grid whose linear index runs over the XCDs first.
// (With no more units than compute units each has one, or nearly, to itself either way.)
static bool spread_batch(const AttnParams& p, int slots) {
  return p.B > 1 && p.B < 65536 && p.H % kNumXcd == 0 && p.n_full == p.total_blocks && 2 * p.total_blocks > slots;
}

// Head size 64 runs three workgroups on a compute unit (kWavesPerSimd): a round of three takes 768 units instead of 512 and, its
// wavefronts covering each other's softmax, less than 1.5 times as long. Where two workgroups need no more rounds than three, two of
// them are faster: units in (768, 1024], two rounds either way, the second one of three partly empty. (Up to 512 units nothing differs.)
// us, two / three, the same bits, bf16:
//   512 units, 8 key tiles 15.4 / 15.2, 64 tiles 76.1 / 76.0     528, 1 tile 10.7 / 8.3     688, 8 tiles 24.3 / 20.4, 86 tiles 170 / 138
//   752, 188 tiles 387 / 307     768, 24 tiles 55.0 / 47.1     776, 16 tiles 41.7 / 43.3, 64 tiles 139 / 148     832, 104 tiles 223 / 238
//   896, 16 tiles 43.0 / 44.4     1024, 16 tiles 45.0 / 45.4, 128 tiles 292 / 300     1200, 32 tiles 106 / 93     1280, 64 tiles 218 / 181
//   1536, 64 tiles 225 / 215     1632, 68 tiles 272 / 261     2048, 8 tiles 53.9 / 48.9     2512, 64 tiles 371 / 353     6144, 8 tiles 162 / 140
// with a mask, f16, every key live: 704, 22 tiles 52.5 / 42.3     800, 20 tiles 53.6 / 56.8     816, 47 tiles 113 / 124     1024, 16 tiles
//   46.8 / 48.2, 64 tiles 162 / 171     1632, 8 tiles 50 / 44.5, 68 tiles 293 / 273     2944, 64 tiles 475 / 436     3072, 16 tiles 143 / 127;
//   one of two rows padded to 40 %, which the launch does not know: 800 units 40.3 / 33.9, 1024 117 / 109, 1632 289 / 271.
// (A unit's first 4 query fragments in LDS and fewer reads ahead, 164 registers: as fast at one round, 1 to 7 % slower beyond.)
// `main_units`: without those that the key split takes. It counts rounds of two (device_slots) in either form, so that what a unit's
// keys are cut into does not depend on the form: us, bf16, split / whole, 520 units of 64 tiles 90 / 97, 640 of 64 113 / 102, of 16
// tiles 47 / 31, 1088 of 64 177 / 169, 1544 of 64 230 / 248, of 16 76 / 71.
static bool fills_two(int64_t main_units, int slots) { return 2 * main_units > 3 * static_cast<int64_t>(slots) && main_units <= 2 * static_cast<int64_t>(slots); }

template <typename T, int D, int NW>
static int launch_dma(AttnParams& p, hipStream_t stream, void* ws, size_t ws_bytes) {
  constexpr int BM = NW * 32;
  p.n_qblocks = (p.Sq + BM - 1) / BM;
  const int64_t total = static_cast<int64_t>(p.n_qblocks) * p.H * p.B;
  if (total > 0x3fffffffll) {
    set_error("odit_attn_fwd: grid of %lld workgroups is too large", static_cast<long long>(total));
    return ODIT_EINVAL;
  }
  p.total_blocks = static_cast<int>(total);
  p.n_full = p.total_blocks; p.key_chunks = 1; p.tiles_per_chunk = 0; p.ws = nullptr;
  p.queue = nullptr; p.epoch = 0;
  TailPlan t{0, 1, 0};
  const int n_tiles = (p.Sk + 63) / 64, slots = device_slots(NW);
  if (ws != nullptr) {
    if ((reinterpret_cast<uintptr_t>(ws) & 15) != 0) {
      set_error("odit_attn_fwd: workspace must be 16-byte aligned");
      return ODIT_EINVAL;
    }
    t = plan_tail(total, n_tiles, slots);
    const size_t need = attn_dma_workspace_bytes(p.B, p.Sq, p.Sk, p.H, D);
    if (ws_bytes < need) {
      set_error("odit_attn_fwd: workspace of %zu bytes given, %zu needed", ws_bytes, need);
      return ODIT_EWORKSPACE;
    }
    if (t.rem > 0) {
      p.n_full = p.total_blocks - t.rem; p.key_chunks = t.key_chunks; p.tiles_per_chunk = t.tiles_per_chunk;
      p.ws = reinterpret_cast<float*>(static_cast<char*>(ws) + kAttnQueueBytes);
    }
  }
  const int n_parts = t.rem * t.key_chunks;
  const bool words = p.mask != nullptr && n_tiles <= kMaskWords;
  int rc = ODIT_OK;
  if (p.n_full > 0) {
    // the persistent form draws its units from ticket words at the head of the workspace
    const int W = (ws != nullptr && NW == 4) ? persistent_workgroups(p.n_full, n_tiles, slots, NW) : 0;
    if constexpr (NW == 4) {
      if (W > 0) {
        p.queue = static_cast<unsigned long long*>(ws);
        p.epoch = next_ticket_epoch() & ((1ull << 40) - 1);
        hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 2>), dim3(W), dim3(NW * 64), 0, stream, p);
      }
    }
    const bool two = D == 64 && NW == 4 && W == 0 && fills_two(p.n_full, slots);
    if constexpr (D == 64 && NW == 4) {
      if (two && words && spread_batch(p, slots))
        hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 8>), dim3(p.n_qblocks * kNumXcd, p.H / kNumXcd, p.B), dim3(NW * 64), 0, stream, p);
      else if (two && words) hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 7>), dim3(p.n_full), dim3(NW * 64), 0, stream, p);
      else if (two) hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 6>), dim3(p.n_full), dim3(NW * 64), 0, stream, p);
    }
    if (W == 0 && !two) {
      if (words && spread_batch(p, slots))
        hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 5>), dim3(p.n_qblocks * kNumXcd, p.H / kNumXcd, p.B), dim3(NW * 64), 0, stream, p);
      else if (words) hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 3>), dim3(p.n_full), dim3(NW * 64), 0, stream, p);
      else hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 0>), dim3(p.n_full), dim3(NW * 64), 0, stream, p);
    }
    rc = check_launch("odit_attn_fwd");
  }
  if (rc != ODIT_OK || n_parts == 0) return rc;
  // stream order puts these after the full rounds, when every slot is free again
  if (words) hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 4>), dim3(n_parts), dim3(NW * 64), 0, stream, p);
  else hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, 1>), dim3(n_parts), dim3(NW * 64), 0, stream, p);
  rc = check_launch("odit_attn_fwd (key-split tail)");
  if (rc != ODIT_OK) return rc;
  const int64_t rows = static_cast<int64_t>(t.rem) * BM;
  hipLaunchKernelGGL((attn_merge_kernel<T, D, BM>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0,
                     stream, p, n_parts);
  return check_launch("odit_attn_fwd (merge)");
}

// Wavefronts per workgroup: 4 (two workgroups per compute unit or, at head size 64, mostly three, each on its own) or 8 (one
// workgroup per compute unit whose two halves run in anti-phase). Side by side in one process when the line was drawn (bf16, us, 4 / 8
// wavefronts, two workgroups of 4 at either head size; two boxes):
//   D=128  B=2 S=4352 H=24  514 / 491, 492 / 473     B=2 S=4096 H=24  429 / 420, 407 / 402
//          B=1 S=4608 H=24  302 / 297, 289 / 288     B=2 S=32760 H=40  38910 / 38616, 37053 / 36483
//   D=64   B=2 S=4352 H=24  326 / 334, 316 / 328
// so head size 128 takes 8 and head size 64 stays at 4 - from 32 key tiles per unit on: the two halves of an
// 8-wavefront workgroup begin and end their unit together, so the unit's fixed cost (first tiles fetched cold,
// first scores, the store) is not hidden behind another workgroup's tiles as it is with two independent workgroups
// per compute unit, and with few tiles per unit that costs more than the anti-phase gains (B=2, 16384 queries,
// 24 heads, 4 / 8 wavefronts: 512 keys 300 / 334 us, 1024 keys 469 / 496, 2048 keys 823 / 823; Wan's cross-attention,
// 32760 queries x 512 keys x 40 heads, 901 / 947). (With the two halves' roles paired wrongly, wavefronts w and
// w + 1 or w and w + 2 in anti-phase instead of w and w + 4, the same kernel is 10 to 18 % slower: two wavefronts of a
// SIMD in the same stage is what costs, and independent workgroups already avoid it most of the time by themselves.)
// Since the softmax's vector work was cut the two are closer, and at head size 128 (us, 4 / 8, the same bits; the largest on another box than the others)
//   from 128 key tiles on 8 are ahead wherever there is a round of units:  B=1 S=8192 H=24 736 / 728, B=2 1475 / 1449, S=16384 H=40 4814 / 4754,
//     B=2 S=32760 H=40 37490 / 37000;
//   below, 4 are, whose units are half as large: of few units every compute unit has one (B=1 S=2100 H=8, 136 units, 41.6 / 54.8, S=4096
//     77.1 / 93.0, 700 queries x 4096 keys H=24 68.6 / 91.3), and a last round is filled better (B=1 H=40 S=2100 105 / 120, B=4 H=16 S=2500
//     210 / 224, B=1 S=3600 H=24 174 / 195, S=6000 H=16 286 / 310, B=2 S=2390 H=24 146 / 151, 16384 queries x 2048 keys H=40 651 / 660);
//   but with more than two rounds of 64 tiles and more it is a draw (B=2 S=4352 H=24 447 / 447, S=4808 552 / 550, S=6032 845 / 858, S=7000 H=40
//     1845 / 1840), in whole steps too: 8. With two rounds or less whole steps are in favour of 4, B=1 S=4608 H=24 alone 256 / 253, in a Flux
//     step 259 / 271, step 0.993; B=1 S=2706 H=40 in a step 0.995;
//   and where 4 put two units of half the size on some compute units in the place of one whole, the anti-phase is 2 to 4 % ahead (units of 4
//     wavefronts above one for each compute unit: B=1 S=5000 H=8, 320 units, 119.6 / 116.2, 1536 queries x 4096 keys H=24, 288, 96.3 / 93.0;
//     cut by keys: 512 x 4096 H=24, 96, 50.0 / 46.4, 256 x 7000 H=40, 80, 59.5 / 54.9). The queries must be whole units of 8 for that: 300 x 4096
//     H=40, 120 units, 50 / 91, 2100 x 2100 H=16, 272, 56.0 / 59.7.
// ODIT_ATTN_WAVES in the environment, read at the first attention launch, overrides the choice (for measurements).
static int dma_waves(int B, int Sq, int Sk, int H, int D) {
  static const int forced = [] {
    const char* e = getenv("ODIT_ATTN_WAVES");
    const int v = e != nullptr ? atoi(e) : 0;
    return (v == 4 || v == 8) ? v : 0;
  }();
  if (forced != 0) return forced;
  const int tiles = (Sk + 63) / 64;
  if (D != 128 || tiles < 32) return 4;
  if (tiles >= 128) return 8;
  const int64_t heads = static_cast<int64_t>(B) * H, units = (Sq + 127) / 128 * heads;
  const int cus = device_slots(8);
  if (tiles >= 64 && units > 4 * cus) return 8;
  const bool whole = 2 * ((Sq + 255) / 256 * heads) == units;
  return whole && ((units > cus && 2 * units <= 3 * cus) || (4 * units > cus && 2 * units <= cus)) ? 8 : 4;
}

size_t attn_dma_workspace_bytes(int B, int Sq, int Sk, int H, int D) {
  if (B <= 0 || Sq <= 0 || Sk <= 0 || H <= 0) return 0;
  const int nw = dma_waves(B, Sq, Sk, H, D);
  const int bm = nw * 32;
  const int64_t units = static_cast<int64_t>((Sq + bm - 1) / bm) * H * B;
  const int n_tiles = (Sk + 63) / 64, slots = device_slots(nw);
  const TailPlan t = plan_tail(units, n_tiles, slots);
  const int64_t main_units = units - t.rem;
  const bool persistent = main_units <= 0x3fffffff && persistent_workgroups(static_cast<int>(main_units), n_tiles, slots, nw) > 0;
  if (t.rem == 0 && !persistent) return 0;
  return kAttnQueueBytes + tail_ws_bytes(t, bm, D);  // ticket words first (zero-filled once), then the tail's partial results
}

// 32-bit buffer offsets: the whole key range of one (batch, head) must be addressable
bool attn_dma_addressable(int Sk, int D, int64_t k_seq_stride, int64_t v_seq_stride) {
  const int64_t k_span = (static_cast<int64_t>(Sk) + 64) * k_seq_stride * 2;
  const int64_t v_span = (static_cast<int64_t>(Sk) + 64) * v_seq_stride * 2;
  // (the tile loads fold their swizzle into the byte offset by an XOR, which needs rows that start on a multiple
  // of their own length of D elements)
  return k_span < (1ll << 31) && v_span < (1ll << 31) && k_seq_stride >= 0 && v_seq_stride >= 0 &&
         k_seq_stride % D == 0 && v_seq_stride % D == 0;
}

int attn_dma_plan(int B, int Sq, int Sk, int H, int D, bool with_workspace, char* text, size_t text_bytes) {
  const int nw = dma_waves(B, Sq, Sk, H, D), bm = nw * 32;
  const int64_t units = static_cast<int64_t>((Sq + bm - 1) / bm) * H * B;
  const int n_tiles = (Sk + 63) / 64, slots = device_slots(nw);
  TailPlan t{0, 1, 0};
  if (with_workspace) t = plan_tail(units, n_tiles, slots);
  // kernel names as a profiler prints them, with T for the element type
  char main_text[160];
  const int64_t main_units = units - t.rem;
  const int W = (!with_workspace || main_units > 0x3fffffff) ? 0 : persistent_workgroups(static_cast<int>(main_units), n_tiles, slots, nw);
  if (W > 0) {
    snprintf(main_text, sizeof(main_text), "attn_fwd_dma_kernel<T, %d, %d, 2> units=%lld on %d persistent workgroups", D,
             nw, static_cast<long long>(main_units), W);
  } else {
    const bool two = D == 64 && nw == 4 && fills_two(main_units, slots);
    snprintf(main_text, sizeof(main_text), "attn_fwd_dma_kernel<T, %d, %d, %d> units=%lld", D, nw, two ? 6 : 0,
             static_cast<long long>(main_units));
  }
  if (t.rem == 0) {
    snprintf(text, text_bytes, "%s", main_text);
    return 1;
  }
  snprintf(text, text_bytes, "%s; attn_fwd_dma_kernel<T, %d, %d, 1> units=%d x %d key ranges of %d tiles; "
           "attn_merge_kernel<T, %d, %d> rows=%d", main_text, D, nw, t.rem, t.key_chunks, t.tiles_per_chunk, D, bm,
           t.rem * bm);
  return main_units > 0 ? 3 : 2;
}

int launch_attn_dma(AttnParams& p, int dtype, int D, hipStream_t stream, void* ws, size_t ws_bytes) {
  if (!attn_dma_addressable(p.Sk, D, p.ks_s, p.vs_s)) return ODIT_ENOTSUP;
#define ODIT_DMA_GO(T)                                                                     \
  if (dma_waves(p.B, p.Sq, p.Sk, p.H, D) == 8) {                                           \
    if (D == 128) return launch_dma<T, 128, 8>(p, stream, ws, ws_bytes);                   \
    return launch_dma<T, 64, 8>(p, stream, ws, ws_bytes);                                  \
  }                                                                                        \
  if (D == 128) return launch_dma<T, 128, 4>(p, stream, ws, ws_bytes);                     \
  return launch_dma<T, 64, 4>(p, stream, ws, ws_bytes);
  if (dtype == ODIT_BF16) { ODIT_DMA_GO(bf16_t) }
  ODIT_DMA_GO(f16_t)
#undef ODIT_DMA_GO
}

}  // namespace odit
