// silu(gate) * up of one element, rounded as F.silu(gate) * up rounds it.
#pragma once

#include "mlr_common.h"

namespace mlr {

template <typename T>
__device__ __forceinline__ T silu_mul_elem(T gate, T up) {
#pragma clang fp contract(off)
  using E = Elem<T>;
  const float g = E::to_f32(gate);
  const T s = E::from_f32(g / (1.0f + expf(-g)));
  return E::from_f32(E::to_f32(s) * E::to_f32(up));
}

}  // namespace mlr
