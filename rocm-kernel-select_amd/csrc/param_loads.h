// Several runtime-typed parameters loaded together.  load_param() branches on the type around each
// load and converts inside the branch, so consecutive calls wait for each load in turn; here the
// branch is taken once and every load is issued before the first conversion.
#pragma once
#include "atk_common.h"

namespace atk {

// o[k] = p[i + k * stride] for k < N
template <int N>
__device__ __forceinline__ void load_params(const void* p, int dtype, int64_t i, int64_t stride, float (&o)[N]) {
  if (dtype == ATK_F32) {
#pragma unroll
    for (int k = 0; k < N; ++k) o[k] = reinterpret_cast<const float*>(p)[i + k * stride];
  } else {
    unsigned short h[N];
#pragma unroll
    for (int k = 0; k < N; ++k) h[k] = reinterpret_cast<const unsigned short*>(p)[i + k * stride];
#pragma unroll
    for (int k = 0; k < N; ++k)
      o[k] = dtype == ATK_F16 ? (float)__builtin_bit_cast(_Float16, h[k]) : (float)__builtin_bit_cast(__bf16, h[k]);
  }
}

}  // namespace atk
