// The gated unit of gated_act.hip and experts.hip.
#pragma once
#include "common_t.h"

// g * sigmoid(alpha (g + cubic g^3)) * (u + offset), g capped at limit, u at +-limit.  QUICK: the
// sigmoid by the hardware's reciprocal (1 ulp, a tenth of the division's instructions), where
// the unit ends a tile of matrix products and nothing else runs beside it
template <bool QUICK = false>
DEV float clamped_glu_f(float g, float u, float limit, float alpha, float offset, float cubic) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  float z = alpha * g;
  if (cubic != 0.f) z *= 1.f + cubic * g * g;
  return g * (QUICK ? __builtin_amdgcn_rcpf(1.f + __expf(-z)) : sigmoid_f(z)) * (u + offset);
}
