// The tile kernel with the order of summation that the library's kernel that is never run would have had where it splits tiles (tile_shares), for calls whose results are
// to be that kernel's. One workgroup sums all pieces of a tile, the sum so far waiting in its scratch: where the pieces ran on several they would have to wait for
// each other. A form of its own, as in the kernels of gemm_tile_apart.hip the tests for it put registers into scratch memory.
#include "gemm_tile.h"

namespace odit {

int launch_gemm_tile_shared(const GemmCall& c, int dtype, const TileShares& shares, void* scratch, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  TilePlan plan;
  plan.bm = 256;
  plan.tiles0 = plan.tiles1 = plan.tiles = plan.whole = shares.tiles;
  plan.parts = 1;
  plan.grid = std::min(shares.tiles, std::min(cus, kGemmMaxWorkers));
  TileArgs<false, false, true> p;
  fill_tile_params(p, plan, &c, 1, nullptr, scratch);
  p.shared = shares.from;
  p.share = shares.share;
  p.more = shares.more;
  const dim3 grid(plan.grid), block(512);
  if (dtype == ODIT_BF16) hipLaunchKernelGGL((gemm_tile_kernel<bf16_t, 4, false, false, true, true>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((gemm_tile_kernel<f16_t, 4, false, false, true, true>), grid, block, 0, stream, p);
  return check_launch("odit_linear (tile kernel)");
}

}  // namespace odit
