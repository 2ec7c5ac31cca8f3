// The kernel for small products (gemm_small.h) with LayerNorm and modulation of its rows in front, the output plain or heads of 64 features.
#include "gemm_small.h"

namespace odit {

template <typename T, bool HEADS>
static void go(const SmallArgs<HEADS, true>& p, unsigned tiles, hipStream_t stream) {
  const dim3 grid(tiles), block(64 * kSmallWaves);
  if (p.k_steps == 1) hipLaunchKernelGGL((gemm_small_kernel<T, 1, HEADS, true>), grid, block, 0, stream, p);
  else if (p.k_steps == 2) hipLaunchKernelGGL((gemm_small_kernel<T, 2, HEADS, true>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((gemm_small_kernel<T, 4, HEADS, true>), grid, block, 0, stream, p);
}

int launch_gemm_small_norm(const GemmCall* c, const RowNorm* norm, const HeadsOut* heads, int dtype, hipStream_t stream) {
  static_assert(kSmallNormK == 4 * kGemmBK, "every step of the reduction has a stage");
  int tiles[2] = {0, 0};
  auto launch = [&](auto& p) {
    fill_small_params(p, c, 2, tiles);
    for (int i = 0; i < 2; ++i) p.norm[i] = norm[i];
    if (dtype == ODIT_BF16) go<bf16_t>(p, tiles[0] + tiles[1], stream);
    else go<f16_t>(p, tiles[0] + tiles[1], stream);
  };
  if (heads != nullptr) {
    SmallArgs<true, true> p;
    for (int i = 0; i < 2; ++i) {
      p.heads[i] = heads[i];
      fill_heads_division(p.heads[i]);
    }
    launch(p);
  } else {
    SmallArgs<false, true> p;
    launch(p);
  }
  return check_launch("odit_linear_pair_norm (small kernel)");
}

}  // namespace odit
