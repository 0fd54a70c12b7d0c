// The experts' activations, the same bits in every form of their products.
#pragma once
#include "common.h"

namespace xi {

template <int ACT>
__device__ __forceinline__ float moe_act_m(float z) {
  if constexpr (ACT == 2) return z > 0.f ? z * z : 0.f;       // the square of relu
  if constexpr (ACT == 0) return z / (1.f + __expf(-z));
  else return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

}  // namespace xi
