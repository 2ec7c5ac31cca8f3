// The rule and the launches of the kernel for small products (the kernel itself: gemm_small.h).
#include "gemm_small.h"

namespace odit {

// Where the kernel is the one to run: every tile has a place at once (as many workgroups to a CU as its LDS holds; a second
// round begins behind the whole latency of the first) and the reduction is short (a step takes 0.25 us). us with the host's part,
// this kernel / stream-K / the library's two launches: M=128+20 N=1024 K=1024 7.8 / 22 / 19; M=128+20 N=512 K=2048 11 / 35 / 19;
// N=1024 K=4096 19 / 26 / 21; two rounds: M=600+77 N=3072 K=1024 21 / 18 / 20, M=600+77 N=4096 K=1024 23 / 23 / 22.
bool gemm_small_rule(const GemmCall* c, int count, int cus, int max_k) {
  const int K = c[0].K, nk = K / kGemmBK;
  if (K > max_k) return false;
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i)
    tiles += static_cast<int64_t>((c[i].M + kSmallTile - 1) / kSmallTile) * ((c[i].N + kSmallTile - 1) / kSmallTile);
  const int per_cu = nk > 4 ? 1 : (nk > 2 ? 2 : 4);  // 160 KB of LDS, and 32 wavefronts
  return tiles <= static_cast<int64_t>(cus) * per_cu;
}

int launch_gemm_small(const GemmCall* c, int count, int dtype, hipStream_t stream) {
  SmallArgs<false, 0> p;
  int tiles[2] = {0, 0};
  fill_small_params(p, c, count, tiles);
  const dim3 grid(tiles[0] + tiles[1]), block(64 * kSmallWaves);
#define ODIT_SMALL(T)                                                                                                    \
  do {                                                                                                                   \
    if (p.k_steps == 1) hipLaunchKernelGGL((gemm_small_kernel<T, 1, false, 0>), grid, block, 0, stream, p);                         \
    else if (p.k_steps == 2) hipLaunchKernelGGL((gemm_small_kernel<T, 2, false, 0>), grid, block, 0, stream, p);                    \
    else if (p.k_steps <= 4) hipLaunchKernelGGL((gemm_small_kernel<T, 4, false, 0>), grid, block, 0, stream, p);                    \
    else hipLaunchKernelGGL((gemm_small_kernel<T, kSmallStages, false, 0>), grid, block, 0, stream, p);                             \
  } while (0)
  if (dtype == ODIT_BF16) ODIT_SMALL(bf16_t);
  else ODIT_SMALL(f16_t);
#undef ODIT_SMALL
  return check_launch("odit_linear (small kernel)");
}

}  // namespace odit
