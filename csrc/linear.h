// Launch arguments of the products of many rows (linear.hip).
#pragma once
#include <hip/hip_runtime.h>

enum LinearUnit { LINEAR_PLAIN, LINEAR_BIAS, LINEAR_SWIGLU, LINEAR_GLU, LINEAR_PARTS };

// y = x w^T (+ bias), or the gated unit of its halves: gates, then ups
struct LinearArgs {
  void* out;         // [M, N], gated [M, N / 2] rows out_stride apart; bf16 like all here
  const void* x;     // [M, K] rows x_stride apart
  const void* w;     // [N, K] rows w_stride apart
  const void* bias;  // [N], LINEAR_BIAS
  int64_t x_stride, w_stride, out_stride;
  int M, N, K;       // K a multiple of 64, outputs of 8; rows 16-byte aligned, operands < 2 GiB
  float limit, alpha, offset, cubic;  // LINEAR_GLU
};

// The tile and the parts of the inner dimension that the sizes call for; unit LINEAR_PARTS: where
// the parts' sums are added up by what reads them
extern "C" void linear_choice(int M, int N, int K, int unit, int* tile, int* splits);
// tile: a number that linear_fits(); from 2 splits on with parts [splits, M, N] fp32, which are
// all that unit LINEAR_PARTS writes
extern "C" void launch_linear(const LinearArgs* a, int unit, int tile, int splits, void* parts,
                              hipStream_t stream);
// Is there such a tile, for gates and ups?
extern "C" bool linear_fits(int tile, bool glu);

// The longest rows that are added up and normed in one pass (elementwise.hip)
#define ADD_RMSNORM_MOST 16384
