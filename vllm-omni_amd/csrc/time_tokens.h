// Launches of the dense projections that end at once where a word on the device says so (time_tokens.hip). `ask`: only whether they can be made.
#pragma once

#include "odit_common.h"

namespace odit {

// linear_few.hip: silu(x) W^T + bias of M dense rows, and odit_time_linear of M timesteps (pre 1), where *only_if is not 0
int linear_few_if(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int dtype, const int* only_if, bool ask,
                  hipStream_t stream);
int time_linear_if(const void* t, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, float neg_log_period, float scale, int t_dtype,
                   int dtype, const int* only_if, bool ask, hipStream_t stream);
// linear.hip: x W^T + bias of M dense rows where *unless is 0, by the tile kernel; ODIT_ENOTSUP where another one is expected to be much faster
int linear_tile_unless(const void* x, const void* w, const void* bias, void* out, int M, int N, int K, int64_t ldw, int dtype, void* workspace,
                       size_t workspace_bytes, const int* unless, bool ask, hipStream_t stream);

}  // namespace odit
