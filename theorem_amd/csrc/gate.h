// Gate arithmetic shared by the chunk-local cumsum (gates.hip) and the chunk
// records (wy_build_A.hip).
#pragma once

#include <math.h>

#include "common.h"

namespace thm {

__device__ __forceinline__ float logsigmoid(float x) {
  // log(sigmoid(x)) = min(x, 0) - log1p(exp(-|x|)), exact in both tails.
  return fminf(x, 0.f) - log1pf(expf(-fabsf(x)));
}

// Inclusive sum over the lanes of a wavefront (lane l: lanes 0 .. l): DPP row
// shifts inside each 16-lane row, then the row totals broadcast upwards.
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, true));
}
__device__ __forceinline__ float wave_inclusive_sum(float v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);  // row_shr:2
  v = dpp_add<0x114, 0xf>(v);  // row_shr:4
  v = dpp_add<0x118, 0xf>(v);  // row_shr:8
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

}  // namespace thm
