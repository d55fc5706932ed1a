// Activation functions in half precision, shared by the kernels that take binary16 tensors.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "sparse_conv_kernels.h"

namespace pl {
namespace half_act {

typedef _Float16 h1;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h1 HalfBits(uint16_t b) { return __builtin_bit_cast(h1, b); }
__device__ __forceinline__ uint16_t BitsOf(h1 v) { return __builtin_bit_cast(uint16_t, v); }
__device__ __forceinline__ h2 Both(h1 v) { return h2{v, v}; }

// Activation on two values, every step its own half-precision instruction:
// relu max(v,0); relu6 min(max(v,0),six); leaky v >= 0 ? v : v*alpha;
// hard_swish (v * (1/scale)) * min(max(v + offset, 0), threshold).
template <int ACT>
__device__ __forceinline__ h2 ActivateH(h2 v, const DevActH& a) {
  const h2 zero = {(h1)0, (h1)0};
  if (ACT == 1) return __builtin_elementwise_max(v, zero);
  if (ACT == 2) return __builtin_elementwise_min(__builtin_elementwise_max(v, zero), Both(HalfBits(a.alpha)));
  if (ACT == 4) {
    const h2 m = v * Both(HalfBits(a.alpha));
    return h2{v.x >= (h1)0 ? v.x : m.x, v.y >= (h1)0 ? v.y : m.y};
  }
  if (ACT == 10) {
    h2 t = v + Both(HalfBits(a.hs_offset));
    const h2 u = v * Both(HalfBits(a.hs_inv_scale));
    t = __builtin_elementwise_min(__builtin_elementwise_max(t, zero), Both(HalfBits(a.hs_threshold)));
    return u * t;
  }
  return v;
}

}  // namespace half_act
}  // namespace pl
