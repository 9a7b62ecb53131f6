// Launch arguments of a side layer's pass (gated_act.hip).
#pragma once
#include <hip/hip_runtime.h>

struct SideLayerArgs {
  float* x;              // [n, w] residual, updated
  const void* y;         // [n, w] bf16, or parts of it [parts, n, w] fp32
  const void* gate;      // [dim, w]
  const void* proj;      // [w, dim]
  const void* table;     // [tokens, dim] rows table_stride apart
  const void* y_norm;    // [w]
  const void* x_norm;    // [w], or null: out is x
  void* out;             // [n, w] rows out_stride apart, or null
  const int64_t* token_ids;
  int64_t table_stride, out_stride;
  int n, w, dim, parts;  // parts 0: y is whole
  float eps;
};
