// The kernel for small products (gemm_small.h) with a norm of its rows in front, the output plain or heads of 64 features.
#include "gemm_small.h"

namespace odit {

template <typename T, bool HEADS, int NORM>
static void go(const SmallArgs<HEADS, NORM>& p, int steps, unsigned tiles, hipStream_t stream) {
  const dim3 grid(tiles), block(64 * kSmallWaves);
  if (steps == 1) hipLaunchKernelGGL((gemm_small_kernel<T, 1, HEADS, NORM>), grid, block, 0, stream, p);
  else if (steps == 2) hipLaunchKernelGGL((gemm_small_kernel<T, 2, HEADS, NORM>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((gemm_small_kernel<T, 4, HEADS, NORM>), grid, block, 0, stream, p);
}

int launch_gemm_small_norm(const GemmCall* c, int count, const RowNorm* norm, const HeadsOut* heads, int dtype, hipStream_t stream) {
  static_assert(kSmallNormK == 4 * kGemmBK, "every step of the reduction has a stage");
  int tiles[2] = {0, 0};
  auto launch = [&](auto& p) {
    fill_small_params(p, c, count, tiles);
    for (int i = 0; i < 2; ++i) p.norm[i] = norm[i < count ? i : 0];
    if (dtype == ODIT_BF16) go<bf16_t>(p, p.k_steps, tiles[0] + tiles[1], stream);
    else go<f16_t>(p, p.k_steps, tiles[0] + tiles[1], stream);
  };
  if (heads != nullptr) {
    SmallArgs<true, kNormAll> p;
    for (int i = 0; i < 2; ++i) {
      p.heads[i] = heads[i];
      fill_heads_division(p.heads[i]);
    }
    launch(p);
  } else {
    SmallArgs<false, kNormAll> p;
    launch(p);
  }
  return check_launch("odit_linear_pair_norm (small kernel)");
}

int launch_gemm_small_stem(const GemmCall* c, const void* weight, float eps, int dtype, hipStream_t stream) {
  SmallArgs<false, kNormStem> p;
  int tiles[2] = {0, 0};
  fill_small_params(p, c, 2, tiles);
  p.weight = weight;
  p.eps = eps;
  p.k_steps1 = c[1].K / kGemmBK;
  const int steps = p.k_steps1 > p.k_steps ? p.k_steps1 : p.k_steps;
  if (dtype == ODIT_BF16) go<bf16_t>(p, steps, tiles[0] + tiles[1], stream);
  else go<f16_t>(p, steps, tiles[0] + tiles[1], stream);
  return check_launch("odit_linear_stem (small kernel)");
}

}  // namespace odit
