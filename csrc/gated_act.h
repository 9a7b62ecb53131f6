// The gated unit of gated_act.hip, latent_proj.hip and experts.hip.
#pragma once
#include "common_t.h"
#include "glu_rows.h"

// g * sigmoid(alpha (g + cubic g^3)) * (u + offset), g capped at limit, u at +-limit
DEV float clamped_glu_f(float g, float u, float limit, float alpha, float offset, float cubic) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  float z = alpha * g;
  if (cubic != 0.f) z *= 1.f + cubic * g * g;
  return g * sigmoid_f(z) * (u + offset);
}

// rows of it, V elements a time: every `step`th from `first` on
template <typename T, int V>
DEV void clamped_glu_rows(const GluRows& a, const int64_t first, const int64_t step) {
  const int per_row = a.inter / V;
  const int64_t total = (int64_t)a.rows * per_row;
  for (int64_t i = first; i < total; i += step) {
    const int64_t r = i / per_row;
    const int c = (int)(i - r * per_row) * V;
    const T* src = (const T*)a.gate_up + r * a.in_stride + c;
    float g[V], u[V];
    load_f<V>(g, src);
    load_f<V>(u, src + a.inter);
#pragma unroll
    for (int k = 0; k < V; ++k) g[k] = clamped_glu_f(g[k], u[k], a.limit, a.alpha, a.offset, a.cubic);
    store_f<V>((T*)a.out + r * a.out_stride + c, g);
  }
}
