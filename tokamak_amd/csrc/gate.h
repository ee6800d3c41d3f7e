#pragma once

#include <hip/hip_runtime.h>

namespace tk {

// act(z) * u behind a product's sums.  0: silu; 1: the tanh form of gelu; 2: with g = min(z, limit), g sigmoid(1.702 g)
// (clamp(u, -limit, limit) + 1).  (A number known to the compiler leaves its form alone.)
__device__ __forceinline__ float gated_value(float z, float u, int act, float limit) {
  if (act == 0) return z / (1.f + __expf(-z)) * u;
  if (act == 1) return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z))) * u;
  const float g = fminf(z, limit);
  return g / (1.f + __expf(-1.702f * g)) * (fminf(fmaxf(u, -limit), limit) + 1.f);
}

// The tanh form of gelu where registers are short: half of z (1 + tanh y) is z / (1 + exp(-2 y)), with no branches for large and small y.
__device__ __forceinline__ float gelu_by_exp(float z, float u) {
  return z / (1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z))) * u;
}

}  // namespace tk
