// The tile kernel with the library's order of operations in its epilogues (gemm_tile.h, APART): for calls whose results are to be those of a
// kernel of the library's that is never run (linear.hip, lin_sound). Kernels of their own, as a choice at a tile's end costs all the others 0.2 to 0.9 % of a model.
#include "gemm_tile.h"

namespace odit {

int launch_gemm_tile_apart(const GemmCall& c, int dtype, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const TilePlan plan = plan_gemm_tile(&c, 1, cus, false);
  TileArgs<false, false> p;
  fill_tile_params(p, plan, &c, 1, nullptr, nullptr);
  const dim3 grid(plan.grid), block(512);
#define ODIT_TILE(T)                                                                                                 \
  do {                                                                                                               \
    if (plan.bm == 256) hipLaunchKernelGGL((gemm_tile_kernel<T, 4, false, false, true>), grid, block, 0, stream, p); \
    else hipLaunchKernelGGL((gemm_tile_kernel<T, 2, false, false, true>), grid, block, 0, stream, p);                \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_TILE(bf16_t);
  else ODIT_TILE(f16_t);
#undef ODIT_TILE
  return check_launch("odit_linear (tile kernel)");
}

}  // namespace odit
