// The kernel for small products (gemm_small.h) with query, key and value heads of 64 features at its end.
#include "gemm_small.h"

namespace odit {

int launch_gemm_small_heads(const GemmCall* c, int count, const HeadsOut* heads, int dtype, hipStream_t stream) {
  SmallArgs<true, 0> p;
  int tiles[2] = {0, 0};
  fill_small_params(p, c, count, tiles);
  for (int i = 0; i < 2; ++i) {
    p.heads[i] = heads[i < count ? i : 0];
    fill_heads_division(p.heads[i]);
  }
  const dim3 grid(tiles[0] + tiles[1]), block(64 * kSmallWaves);
#define ODIT_SMALL(T)                                                                                                     \
  do {                                                                                                                    \
    if (p.k_steps == 1) hipLaunchKernelGGL((gemm_small_kernel<T, 1, true, 0>), grid, block, 0, stream, p);                    \
    else if (p.k_steps == 2) hipLaunchKernelGGL((gemm_small_kernel<T, 2, true, 0>), grid, block, 0, stream, p);               \
    else if (p.k_steps <= 4) hipLaunchKernelGGL((gemm_small_kernel<T, 4, true, 0>), grid, block, 0, stream, p);               \
    else hipLaunchKernelGGL((gemm_small_kernel<T, kSmallStages, true, 0>), grid, block, 0, stream, p);                        \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_SMALL(bf16_t);
  else ODIT_SMALL(f16_t);
#undef ODIT_SMALL
  return check_launch("odit_linear_heads (small kernel)");
}

}  // namespace odit
