// Rows of a gated unit: [gate | up] -> out (gated_act.h).
#pragma once
#include <cstdint>

struct GluRows {
  void* out;            // [rows, inter]
  const void* gate_up;  // [rows, 2 inter]
  int64_t in_stride, out_stride;
  int rows, inter;
  float limit, alpha, offset, cubic;

  // workgroups of 256 threads that do V elements to a thread, or a share of more than that
  int blocks(int v, int most) const {
    const int64_t want = ((int64_t)rows * (inter / v) + 255) / 256;
    return (int)(want < most ? want : most);
  }
};
