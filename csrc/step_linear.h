// Launch arguments of the projections of a small decode step (step_linear.hip).
#pragma once
#include <hip/hip_runtime.h>

#define STEP_LINEAR_ROWS 4

struct StepLinearArgs {
  void* out;         // [M, N], GLU [M, N / 2]; bf16 like all here
  const void* x;     // [M, K] rows x_stride apart
  const void* w;     // [N, K] rows w_stride apart; GLU: gates, then ups
  const void* bias;  // [N] or null
  int64_t x_stride, w_stride;
  int M, N, K;       // M at most STEP_LINEAR_ROWS, K a multiple of 32; rows 16-byte aligned
};

extern "C" void launch_step_linear(const StepLinearArgs* a, bool glu, hipStream_t stream);
