// The cosine and sine of a timestep at one frequency, as every kernel that forms them does it.
#pragma once

#include "odit_common.h"

namespace odit {

// cos | sin of scale * (t * exp(neg_log_period j / half)); the accurate exp, cos and sin, which torch calls.
// `pre` other than 1 is a factor that the caller's expression applies in T before it (Flux: timestep.to(T) * 1000).
template <typename T, typename TT>
__device__ __forceinline__ void time_sinusoid(TT t, int j, int half, float neg_log_period, float scale, float pre, T& c, T& s) {
#pragma clang fp contract(off)
  const float freq = expf(neg_log_period * static_cast<float>(j) / static_cast<float>(half));
  float tv = to_float(t);
  if (pre != 1.f) tv = round_to<T>(round_to<T>(tv) * pre);
  const float arg = scale * (tv * freq);
  c = from_float<T>(cosf(arg));
  s = from_float<T>(sinf(arg));
}

}  // namespace odit
