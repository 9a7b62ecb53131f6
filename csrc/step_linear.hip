// y = x w^T (+ bias) for the at most four rows of a small decode step (gfx950); GLU: the two
// halves of y as silu(gate) * up, without a pass of its own.
//
// Bound by reading every weight once.  A workgroup owns 16 outputs (GLU: 16 gates and their
// ups) for all rows; its waves split the inner dimension, so that every launch has all CUs
// reading.  Weights go straight from memory, past the caches, to the matrix cores (16x16x32), 8
// rows of a whole line (64 inner elements) a load: the lanes' upper 8 rows of a product are the
// same weights' rows with the line's other half, and so are the upper 8 columns for x.  Of a
// product's results those count whose row and column have the same half; the halves' and
// the waves' sums meet in LDS, in a fixed order, in fp32.
//
// With 16 rows of half a line a load, whose other half came with the next, this took 1.05 to 1.35
// times as long; a quarter of the rows by two lines a load is slower than either.  One row, every
// weight from memory, us, before, now, and the GEMM library (with the GLU's own pass): 28672 x 4096
// GLU 51 41 66, 22016 x 4096 GLU 39 29 52, 6144 x 4096 13.8 12.0 15.5, 4096 x 4096 8.4 8.0 15.6, 4096 x
// 14336 26.7 20.4 25.2, 128256 x 4096 186 156 184, 20048 x 2048 22.3 16.2 49.
// 16 waves and 4 lines in flight each, or for the GLU 8 and 2 of both: 8 waves 1 to 10% slower at
// 6144 x 4096 and above without the GLU, 4 waves 40% slower at 4096 outputs.
#include <type_traits>

#include "common_t.h"
#include "step_linear.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

template <bool GLU, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void step_linear_kernel(const StepLinearArgs a) {
  constexpr int NT = GLU ? 2 : 1;
  constexpr int DEEP = 4 / NT;  // lines of a row whose loads are in flight together
  __shared__ float sums[WAVES][2][NT][16][STEP_LINEAR_ROWS];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 7, half = lane >> 3 & 1, j = lane >> 4;
  const int outs = GLU ? a.N / 2 : a.N, o0 = blockIdx.x * 16;
  const int lines = a.K / 64, each = (lines + WAVES - 1) / WAVES;
  const int s1 = min(lines, (wid + 1) * each);

  const int in = half * 32 + j * 8;  // of a line
  const bf16_t* const xr = (const bf16_t*)a.x + (int64_t)min(c, a.M - 1) * a.x_stride + in;
  const bf16_t* wr[NT][2];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int p = 0; p < 2; ++p)
      wr[n][p] = (const bf16_t*)a.w + (int64_t)(min(o0 + 8 * p + c, outs - 1) + n * outs) * a.w_stride + in;
  f32x4_v acc[NT][2] = {};
  auto some = [&](int s, auto count) {
    constexpr int C = decltype(count)::value;
    bf16x8_v w[C][NT][2], x[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          w[i][n][p] = __builtin_nontemporal_load((const bf16x8_v*)(wr[n][p] + (s + i) * 64));
      x[i] = *(const bf16x8_v*)(xr + (s + i) * 64);
    }
#pragma unroll
    for (int i = 0; i < C; ++i)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          acc[n][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][n][p], x[i], acc[n][p], 0, 0, 0);
  };
  int s = wid * each;
  for (; s + DEEP <= s1; s += DEEP) some(s, std::integral_constant<int, DEEP>());
  for (; s < s1; ++s) some(s, std::integral_constant<int, 1>());
  if (a.K % 64 && wid == WAVES - 1) {  // half a line
    bf16x8_v x = {};
    if (!half) x = *(const bf16x8_v*)(xr + lines * 64);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        bf16x8_v w = {};
        if (!half) w = *(const bf16x8_v*)(wr[n][p] + lines * 64);
        acc[n][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc[n][p], 0, 0, 0);
      }
  }

  // a lane has a product's rows 4 j .. 4 j + 3, so the half j / 2, of its column
  if (c < a.M && half == j >> 1) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[wid][half][n][8 * p + 4 * (j & 1) + r][c] = acc[n][p][r];
  }
  __syncthreads();
  const int row = threadIdx.x >> 4, o = threadIdx.x & 15;
  if (row >= a.M || o0 + o >= outs) return;
  float v[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    v[n] = a.bias ? bf2f(((const bf16_t*)a.bias)[o0 + o + n * outs]) : 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[n] += sums[w][0][n][o][row] + sums[w][1][n][o][row];
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
  const dim3 grid((outs + 15) / 16);
  if (glu)
    step_linear_kernel<true, 8><<<grid, 64 * 8, 0, stream>>>(*a);
  else
    step_linear_kernel<false, 16><<<grid, 64 * 16, 0, stream>>>(*a);
}
