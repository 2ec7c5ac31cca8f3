// The tile kernel's plan and launches (the kernel itself: gemm_tile.h).
#include "gemm_tile.h"

namespace odit {

bool gemm_tile_takes(const GemmCall& c, int dtype) {
  if (dtype != ODIT_BF16 && dtype != ODIT_F16) return false;
  // (8 rows: what is fetched behind the last segment stays inside the operands)
  if (c.M < 8 || c.K < kTileK || c.K % kTileK != 0 || c.N < 8 || c.N % 8 != 0) return false;
  if (c.ldx % 8 != 0 || c.ldw % 8 != 0 || c.ldo % 8 != 0) return false;
  if (!aligned16(c.x) || !aligned16(c.w) || !aligned16(c.out)) return false;
  if (c.bias != nullptr && !aligned16(c.bias)) return false;
  const bool gated = c.epilogue == ODIT_EPI_GATED_RESIDUAL || c.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE;
  if (gated) {
    if (c.residual == nullptr || c.ldr % 8 != 0 || !aligned16(c.residual)) return false;
    if (c.gate != nullptr && (!aligned16(c.gate) || c.ldg % 8 != 0)) return false;
    if (c.epilogue == ODIT_EPI_GATED_RESIDUAL_PRE && !c.gate_f32) return false;
  }
  // 32-bit byte offsets
  const uint64_t xb = (static_cast<uint64_t>(c.M - 1) * c.ldx + c.K) * 2, wb = (static_cast<uint64_t>(c.N - 1) * c.ldw + c.K) * 2;
  if (xb >= (1ull << 32) || wb >= (1ull << 32)) return false;
  return static_cast<int64_t>(row_tiles(c.M, 128)) * row_tiles(c.N, kTileN) < (1 << 28);
}

// Tile height, and whether and into how many parts the tiles of the last round are cut: by expected time, fitted to 268
// launches of 256 to 9500 rows of the projections of widths 3072 and 5120, those within a quarter of a problem's best (6.3 %;
// choosing by it takes 0.2 % longer than the best of all plans). A step takes 1.22 us on 256-row tiles in a launch's first
// round, 1.32 in later ones (the clock falls), 1.13 where a round is cut, 0.78 on 128-row tiles; a launch 3.1, a tile's end 5.7,
// 3 (2) more with GELU; a cut 0.088 for each part (0.057 with 128 rows), 5.7 more behind whole tiles, and 0.2 for every part of a tile beyond four, of
// which there are none behind whole tiles (M=640, N=15360, K=5120: 128 rows in 5 parts 111, 256 rows whole 98; N=13824 8 parts 104, whole 95). M=459, N=5120, K=13824: 256
// rows in 4 parts 80 us, 3 parts 98, 2 parts 131, whole 238, 128 rows in 3 parts 77, 2 parts 100; M=504, N=9216, K=3072: 256
// rows in 3 parts 41, whole 64, 128 rows 48; M=2998, N=12288, K=3072 with GELU: 256 rows in 4 parts 184, whole 215.
TilePlan plan_gemm_tile(const GemmCall* c, int count, int cus, bool scratch) {
  TilePlan best;
  const int most = cus < kGemmMaxWorkers ? cus : kGemmMaxWorkers, nk = c[0].K / kTileK;
  for (int bm = 256; bm >= 128; bm /= 2) {
    const bool tall = bm == 256;
    TilePlan p;
    p.bm = bm;
    p.tiles0 = row_tiles(c[0].M, bm) * row_tiles(c[0].N, kTileN);
    p.tiles1 = p.tiles0 + (count > 1 ? row_tiles(c[1].M, bm) * row_tiles(c[1].N, kTileN) : 0);
    p.tiles = p.tiles1 + (count > 2 ? row_tiles(c[2].M, bm) * row_tiles(c[2].N, kTileN) : 0);
    const int rounds = p.tiles / most, rest = p.tiles - rounds * most;
    float end = 5.7f;
    for (int i = 0; i < count; ++i)
      if (c[i].epilogue == ODIT_EPI_GELU_TANH || c[i].epilogue == ODIT_EPI_BIAS_GELU_TANH) end = tall ? 8.7f : 7.7f;
    auto whole_rounds = [&](int n) { return n == 0 ? 0.f : n * (nk * (tall ? 1.32f : .78f) + end) - nk * (tall ? .1f : 0.f); };
    for (int parts = 1; parts <= kMaxParts[tall]; ++parts) {
      if (parts > 1 && (!scratch || rest == 0 || rest * parts > most || parts > nk || (rounds > 0 && parts > 4))) break;
      p.parts = parts;
      p.whole = parts > 1 ? p.tiles - rest : p.tiles;
      p.grid = rounds > 0 ? most : rest * parts;
      if (parts == 1) {
        p.us = 3.1f + whole_rounds(rounds + (rest > 0 ? 1 : 0));
      } else {
        p.us = 3.1f + whole_rounds(rounds) + (nk + parts - 1) / parts * (tall ? 1.13f : .78f) + rest * parts * (tall ? .088f : .057f) +
               (rounds > 0 ? 5.7f : 0.f) + (parts > 4 ? .2f * (parts - 4) : 0.f);
      }
      if (best.bm == 0 || p.us < best.us) best = p;
    }
  }
  return best;
}

int launch_gemm_tile(const GemmCall* c, int count, const TileX2* x2, int dtype, void* scratch, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const TilePlan plan = plan_gemm_tile(c, count, cus, scratch != nullptr);
  TileArgs<false, false> p;
  fill_tile_params(p, plan, c, count, x2, scratch);
  const dim3 grid(plan.grid), block(512);
#define ODIT_TILE(T)                                                                          \
  do {                                                                                        \
    if (plan.bm == 256) hipLaunchKernelGGL((gemm_tile_kernel<T, 4, false, false>), grid, block, 0, stream, p); \
    else hipLaunchKernelGGL((gemm_tile_kernel<T, 2, false, false>), grid, block, 0, stream, p);              \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_TILE(bf16_t);
  else ODIT_TILE(f16_t);
#undef ODIT_TILE
  return check_launch("odit_linear (tile kernel)");
}

}  // namespace odit
