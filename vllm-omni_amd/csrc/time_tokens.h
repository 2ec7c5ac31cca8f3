// Launches of the dense projections that do the one thing or the other by a word on the device (time_tokens.hip). `ask`: only whether they can be made.
#pragma once

#include "odit_common.h"

namespace odit {

// What a launch for few rows does in their place where *few is 0: `out` = silu of `n` 16-byte vectors x (linear_few_or); the rows [n, K] of timesteps
// x [n] of t_dtype to `out`, or nothing where that is null (time_linear_or).
struct FewOr {
  const int* few;
  const void* x;
  void* out;
  int64_t n;
};
// linear_few.hip: silu(x) W^T + bias of M dense rows, and odit_time_linear of M timesteps (pre 1), where *other.few is not 0
int linear_few_or(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int dtype, const FewOr& other, bool ask,
                  hipStream_t stream);
int time_linear_or(const void* t, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, float neg_log_period, float scale, int t_dtype,
                   int dtype, const FewOr& other, bool ask, hipStream_t stream);
// linear.hip: x W^T + bias of M dense rows where *unless is 0, by the tile kernel; ODIT_ENOTSUP where another one is expected to be much faster
int linear_tile_unless(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int dtype, void* workspace,
                       size_t workspace_bytes, const int* unless, bool ask, hipStream_t stream);

}  // namespace odit
