// The tile kernel for a launch whose work another one may have made unnecessary (gemm_tile.h, UNLESS).
#include "gemm_tile.h"

namespace odit {

int launch_gemm_tile_unless(const GemmCall& c, const int* unless, int dtype, void* scratch, hipStream_t stream) {
  const int cus = device_cus();
  if (cus <= 0) { set_error("odit_linear: cannot read the device's compute-unit count"); return ODIT_ELAUNCH; }
  const TilePlan plan = plan_gemm_tile(&c, 1, cus, scratch != nullptr);
  TileArgs<false, true> p;
  fill_tile_params(p, plan, &c, 1, nullptr, scratch);
  p.unless = unless;
  const dim3 grid(plan.grid), block(512);
#define ODIT_TILE(T)                                                                                      \
  do {                                                                                                    \
    if (plan.bm == 256) hipLaunchKernelGGL((gemm_tile_kernel<T, 4, false, true>), grid, block, 0, stream, p); \
    else hipLaunchKernelGGL((gemm_tile_kernel<T, 2, false, true>), grid, block, 0, stream, p);              \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_TILE(bf16_t);
  else ODIT_TILE(f16_t);
#undef ODIT_TILE
  return check_launch("odit_time_tokens (tile kernel)");
}

}  // namespace odit
