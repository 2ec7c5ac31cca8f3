// The tile kernel for projections to query, key and value heads (gemm_tile.h, HEADS): norm over each head, rotation and the joint
// sequence's layout at the tile's end, in the place of a pass over the projection's output.
#include "gemm_tile.h"

namespace odit {

bool gemm_tile_heads_takes(const GemmCall& c, const HeadsOut& h) {
  // (a wavefront's 32 features are one head's, four wavefronts' 128 are one or two heads; 32-bit divisions of row numbers)
  return (h.D == 64 || h.D == 128) && c.N == 3 * h.HD && h.HD % h.D == 0 && h.S > 0 && (c.epilogue == ODIT_EPI_NONE || c.epilogue == ODIT_EPI_BIAS) &&
         h.k != nullptr && h.v != nullptr && h.wq != nullptr && h.wk != nullptr && h.cos != nullptr && h.sin != nullptr && aligned16(h.q) &&
         aligned16(h.k) && aligned16(h.v) && aligned16(h.wq) && aligned16(h.wk) && aligned16(h.cos) && aligned16(h.sin);
}

int launch_gemm_tile_heads(const GemmCall* c, int count, const HeadsOut* heads, int dtype, void* scratch, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear_heads: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const TilePlan plan = plan_gemm_tile(c, count, cus, scratch != nullptr);
  TileArgs<true, false> p;
  fill_tile_params(p, plan, c, count, nullptr, scratch);
  for (int i = 0; i < 2; ++i) {
    HeadsOut& h = p.heads[i];
    h = heads[i < count ? i : 0];
    fill_heads_division(h);
  }
  const dim3 grid(plan.grid), block(512);
#define ODIT_TILE(T)                                                                                \
  do {                                                                                              \
    if (plan.bm == 256) hipLaunchKernelGGL((gemm_tile_kernel<T, 4, true, false>), grid, block, 0, stream, p); \
    else hipLaunchKernelGGL((gemm_tile_kernel<T, 2, true, false>), grid, block, 0, stream, p);              \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_TILE(bf16_t);
  else ODIT_TILE(f16_t);
#undef ODIT_TILE
  return check_launch("odit_linear_heads (tile kernel)");
}

}  // namespace odit
