// y = x w^T (+ bias) for the at most four rows of a small decode step (gfx950); GLU: the two
// halves of y as silu(gate) * up, without a pass of its own.
//
// Bound by reading every weight once.  A workgroup owns 16 outputs (GLU: 16 gates and their
// ups) for all rows; its 8 waves split the inner dimension, so that every launch has all CUs
// reading.  Weights go straight from memory to the matrix cores (16x16x32, A = 16 rows of
// weights, 8 inner elements a lane) with 16 KiB of a wave's loads in flight, and the rows of x
// from L2 in the same form (B; lanes past the last row read it again).  The waves' sums meet in
// LDS, in a fixed order, in fp32.
//
// One row, against the GEMM library (and the GLU's own pass) before, us, every weight from
// memory: 28672 x 4096 GLU 54 (64), 22016 x 4096 GLU 41 (54), 6144 x 4096 14.0 (14.7), 4096 x 4096
// 8.5 (15.6), 20048 x 2048 22 (50), 2048 x 2048 5.2 (11.0).  384 workgroups (6144 outputs) leave
// half of the CUs with one and half with two.
// Half and twice the loads in flight, 4 and 16 waves, the next group's loads during a group's
// products, 32 outputs a workgroup: all slower by 2 to 40% at most of these sizes.
#include <type_traits>

#include "common_t.h"
#include "step_linear.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

#define WAVES 8

template <bool GLU>
__global__ __launch_bounds__(64 * WAVES) void step_linear_kernel(const StepLinearArgs a) {
  constexpr int NT = GLU ? 2 : 1;
  constexpr int DEEP = 16 / NT;  // steps of 32 whose loads are in flight together
  __shared__ float sums[WAVES][NT][16][STEP_LINEAR_ROWS];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, j = lane >> 4;
  const int outs = GLU ? a.N / 2 : a.N, o0 = blockIdx.x * 16;
  const int steps = a.K / 32, each = (steps + WAVES - 1) / WAVES;
  const int s1 = min(steps, (wid + 1) * each);

  const bf16_t* const xr = (const bf16_t*)a.x + (int64_t)min(c, a.M - 1) * a.x_stride + j * 8;
  const bf16_t* wr[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
    wr[n] = (const bf16_t*)a.w + (int64_t)(min(o0 + c, outs - 1) + n * outs) * a.w_stride + j * 8;
  f32x4_v acc[NT] = {};
  auto some = [&](int s, auto count) {
    constexpr int C = decltype(count)::value;
    bf16x8_v w[C][NT], x[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
#pragma unroll
      for (int n = 0; n < NT; ++n)
        w[i][n] = __builtin_nontemporal_load((const bf16x8_v*)(wr[n] + (s + i) * 32));
      x[i] = *(const bf16x8_v*)(xr + (s + i) * 32);
    }
#pragma unroll
    for (int i = 0; i < C; ++i)
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][n], x[i], acc[n], 0, 0, 0);
  };
  int s = wid * each;
  for (; s + DEEP <= s1; s += DEEP) some(s, std::integral_constant<int, DEEP>());
  for (; s + 4 <= s1; s += 4) some(s, std::integral_constant<int, 4>());
  for (; s < s1; ++s) some(s, std::integral_constant<int, 1>());

  // a lane has outputs 4 j .. 4 j + 3 of row c
  if (c < a.M) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) sums[wid][n][4 * j + r][c] = acc[n][r];
  }
  __syncthreads();
  const int row = threadIdx.x >> 4, o = threadIdx.x & 15;
  if (row >= a.M || o0 + o >= outs) return;
  float v[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    v[n] = a.bias ? bf2f(((const bf16_t*)a.bias)[o0 + o + n * outs]) : 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[n] += sums[w][n][o][row];
  }
  bf16_t* dst = (bf16_t*)a.out + (int64_t)row * outs + o0 + o;
  if constexpr (GLU) {
    // both rounded, as they are between two passes
    const float g = bf2f(f2bf(v[0])), u = bf2f(f2bf(v[NT - 1]));
    *dst = f2bf(g / (1.f + __expf(-g)) * u);
  } else {
    *dst = f2bf(v[0]);
  }
}

extern "C" void launch_step_linear(const StepLinearArgs* a, bool glu, hipStream_t stream) {
  const int outs = glu ? a->N / 2 : a->N;
  auto k = glu ? step_linear_kernel<true> : step_linear_kernel<false>;
  k<<<dim3((outs + 15) / 16), 64 * WAVES, 0, stream>>>(*a);
}
