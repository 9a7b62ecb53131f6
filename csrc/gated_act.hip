// Gated activations over row-strided GEMM outputs (gfx950).
//
//   clamped_glu: g = min(gate, limit), u = clamp(up, +-limit);
//                g * sigmoid(alpha (g + cubic g^3)) * (u + offset)
//   gelu_gate:   gelu_tanh(s) * table[token, offset + i]
//   side_gate:   x + y, then gelu_gate of (gate x): for few tokens, where two
//                elementwise launches and a GEMM of one narrow tile cost more than
//                reading the small weight once per token from L2
//   side_layer: all that a side layer does to one token's row, in one launch
#include <type_traits>

#include "common_t.h"
#include "gated_act.h"
#include "launch.h"
#include "side_layer.h"

template <typename T, int V>
__global__ __launch_bounds__(256) void clamped_glu_kernel(const GluRows a) {
  clamped_glu_rows<T, V>(a, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256);
}

DEV float gelu_tanh_f(float z) {
  return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// Workgroups (token, part of the outputs); the new residual row waits in LDS, in
// the GEMM's input precision, for its dot products.  Every part sums the row, one
// writes it: to a new residual, since the others may still be reading the old.
// All its loads are issued far ahead of their use: one token's latency is the cost.
template <typename T, int V>
__global__ __launch_bounds__(512) void side_gate_kernel(
    float* __restrict__ x_out, const float* __restrict__ x, const T* __restrict__ y,
    const T* __restrict__ gate, const int64_t* __restrict__ token_ids,
    const T* __restrict__ table, T* __restrict__ s, const int w, const int dim,
    const int64_t table_stride) {
  extern __shared__ char lds_raw[];
  T* row = (T*)lds_raw;
  const int64_t n = blockIdx.x;
  const int lane = threadIdx.x & 63;
  // a wave's two outputs; lane j keeps output j's table entry
  const int o0 = (blockIdx.y * 8 + (threadIdx.x >> 6)) * 2;
  const int oj = o0 + (lane & 1);
  const float e = oj < dim ? to_f(table[token_ids[n] * table_stride + oj]) : 0.f;
#pragma unroll 4
  for (int i = threadIdx.x * 4; i < w; i += 2048) {
    float a[4], b[4];
    load_f<4>(a, x + n * w + i);
    load_f<4>(b, y + n * w + i);
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] += b[k];
    if (blockIdx.y == 0) store_f<4>(x_out + n * w + i, a);
    store_f<4>(row + i, a);
  }
  __syncthreads();
  if (o0 >= dim) return;
  const T* g0 = gate + (int64_t)o0 * w;
  const T* g1 = gate + (int64_t)min(o0 + 1, dim - 1) * w;
  float acc0 = 0.f, acc1 = 0.f;
#pragma unroll 8
  for (int i = lane * V; i < w; i += 64 * V) {
    float v[V], p[V], q[V];
    load_f<V>(p, g0 + i);
    load_f<V>(q, g1 + i);
    load_f<V>(v, row + i);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      acc0 += p[k] * v[k];
      acc1 += q[k] * v[k];
    }
  }
  acc0 = wave_sum(acc0);
  acc1 = wave_sum(acc1);
  // the product is an activation: model precision, as a GEMM would store it
  const float z = to_f(from_f<T>(lane & 1 ? acc1 : acc0));
  if (lane < 2 && oj < dim) s[n * dim + oj] = from_f<T>(gelu_tanh_f(z) * e);
}

// sum of LANES neighbours, to each of them
template <int LANES>
DEV float lanes_sum(float v) {
  v = dpp_add<0xb1>(v);  // quad_perm: the other of a pair
  v = dpp_add<0x4e>(v);  // the other pair
  if constexpr (LANES >= 8) v = dpp_add<0x141>(v);   // row_half_mirror
  if constexpr (LANES >= 16) v = dpp_add<0x140>(v);  // row_mirror
  return v;
}

DEV float wave_sum_rows(float v) {
  v = row16_sum(v);
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// of 16 waves, to each thread
DEV float sum_of_1024(float v, float* scratch) {
  v = wave_sum_rows(v);
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return row16_sum(scratch[threadIdx.x & 15]);
}

// x += y; x += rmsnorm(proj (gelu_gate(gate x))) * y_norm; out = layernorm(x) * x_norm, of one token: y in
// 16 bits or as the parts of a product, which are added up in their order; with every rounding
// that the passes by themselves have.  A workgroup reads both weights whole, 512 KB at a width of 2048 and
// 64 outputs, and waits for its loads: those of a phase are on their way before the barrier that it begins with,
// and a wave's lanes read neighbouring bytes of both.  40 tokens: 13.0 us (18.1 with a row of proj to a lane, as
// its lines did not stay in the L1), before, by the sum of the parts (4.8), side_gate (5.7), a product of the
// library (4.9) and residual_norm (5.2), 20.6 and three gaps between launches.
template <int R>  // outputs of a wave
__global__ __launch_bounds__(1024) void side_layer_kernel(const SideLayerArgs a) {
  constexpr int G = 2 * R;              // lanes to a row of proj
  constexpr int CH = R > 4 ? 2 : 4;     // pieces of 512 columns of the gate at once
  constexpr int PR = 8;                 // loads of proj at once
  extern __shared__ float lds[];
  const int w = a.w, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t n = blockIdx.x;
  float* const row = lds;                       // [w] x, then with what is added
  bf16_t* const h = (bf16_t*)(row + w);         // [w]
  float* const s = (float*)(h + w);             // [16 R]
  float* const scratch = s + 16 * R;            // [3][16]
  float* const x = a.x + n * w;
  Pack<bf16_t, 8> gate[CH][R], proj[PR];
  auto load_gate = [&](int from) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int r = 0; r < R; ++r)
        gate[c][r] = *(const Pack<bf16_t, 8>*)((const bf16_t*)a.gate +
            (int64_t)min(wid * R + r, a.dim - 1) * w + min(from + c * 512 + lane * 8, w - 8));
  };
  const int k0 = min(lane % G * 8, a.dim - 8);
  auto output = [&](int i) { return (i * 16 + wid) * (64 / G) + lane / G; };
  auto load_proj = [&](int from) {
#pragma unroll
    for (int i = 0; i < PR; ++i)
      proj[i] = *(const Pack<bf16_t, 8>*)((const bf16_t*)a.proj + (int64_t)min(output(from + i), w - 1) * a.dim + k0);
  };

  const int oj = min(wid * R + lane, a.dim - 1);  // lane j keeps output j's table entry
  const float e = lane < R ? to_f(((const bf16_t*)a.table)[a.token_ids[n] * a.table_stride + oj]) : 0.f;
  load_gate(0);
  for (int i = tid * 4; i < w; i += 4096) {
    float t[4], y[4] = {};
    load_f<4>(t, x + i);
    if (a.parts) {
      const float* from = (const float*)a.y + n * w + i;
#pragma unroll 4
      for (int p = 0; p < a.parts; ++p) {
        float v[4];
        load_f<4>(v, from + (int64_t)p * a.n * w);
#pragma unroll
        for (int k = 0; k < 4; ++k) y[k] += v[k];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = to_f(from_f<bf16_t>(y[k]));
    } else {
      load_f<4>(y, (const bf16_t*)a.y + n * w + i);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] += y[k];
    store_f<4>(row + i, t);
    store_f<4>(h + i, t);
  }
  __syncthreads();

  float acc[R] = {};
  for (int from = 0; from < w; from += CH * 512) {
    if (from) load_gate(from);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = from + c * 512 + lane * 8;
      if (i >= w) continue;
      float v[8];
      load_f<8>(v, h + i);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[r] += to_f(gate[c][r].v[k]) * v[k];
    }
  }
  load_proj(0);
  Pack<bf16_t, 4> y_norm, x_norm;
  auto load_norm = [&](Pack<bf16_t, 4>& g, const void* from, int i) {
    g = *(const Pack<bf16_t, 4>*)((const bf16_t*)from + i);
  };
  load_norm(y_norm, a.y_norm, min(tid * 4, w - 4));
  if (a.x_norm) load_norm(x_norm, a.x_norm, min(tid * 4, w - 4));
  float z = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float sum = wave_sum_rows(acc[r]);
    z = lane == r ? sum : z;
  }
  // products are activations: in the model's precision
  if (lane < R) {
    z = to_f(from_f<bf16_t>(z));
    s[wid * R + lane] = wid * R + lane < a.dim ? to_f(from_f<bf16_t>(gelu_tanh_f(z) * e)) : 0.f;
  }
  __syncthreads();

  bf16_t* const y = h;  // which all waves have read
  float ss = 0.f, sv[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) sv[k] = s[k0 + k];
  const bool counts = lane % G * 8 < a.dim;
  for (int from = 0; output(from) - lane / G < w; from += PR) {
    if (from) load_proj(from);
#pragma unroll
    for (int i = 0; i < PR; ++i) {
      float sum = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) sum += to_f(proj[i].v[k]) * sv[k];
      const bf16_t r = from_f<bf16_t>(lanes_sum<G>(counts ? sum : 0.f));
      const int o = output(from + i);
      if (lane % G == 0 && o < w) {
        y[o] = r;
        ss += to_f(r) * to_f(r);
      }
    }
  }
  const float scale = rsqrtf(sum_of_1024(ss, scratch) / w + a.eps);  // and a barrier
  float sum = 0.f;
  for (int i = tid * 4; i < w; i += 4096) {
    float t[4], d[4];
    load_f<4>(t, row + i);
    load_f<4>(d, y + i);
    if (i >= 4096) load_norm(y_norm, a.y_norm, i);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      t[k] += to_f(y_norm.v[k]) * d[k] * scale;
      sum += t[k];
    }
    store_f<4>(x + i, t);
    store_f<4>(row + i, t);
  }
  if (!a.out) return;
  float mean = 0.f, inv = 1.f;
  if (a.x_norm) {
    mean = sum_of_1024(sum, scratch + 16) / w;
    float sq = 0.f;
    for (int i = tid * 4; i < w; i += 4096)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float c = row[i + k] - mean;
        sq += c * c;
      }
    inv = rsqrtf(sum_of_1024(sq, scratch + 32) / w + a.eps);
  }
  for (int i = tid * 4; i < w; i += 4096) {
    float t[4];
    load_f<4>(t, row + i);
    if (a.x_norm && i >= 4096) load_norm(x_norm, a.x_norm, i);
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] = (t[k] - mean) * inv * (a.x_norm ? to_f(x_norm.v[k]) : 1.f);
    store_f<4>((bf16_t*)a.out + n * a.out_stride + i, t);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void gelu_gate_kernel(
    T* __restrict__ s, const int64_t* __restrict__ token_ids,
    const T* __restrict__ table, const int dim, const int64_t total,
    const int64_t table_stride) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t r = i / dim;
  const float e = to_f(table[token_ids[r] * table_stride + (i - r * dim)]);
  s[i] = from_f<T>(gelu_tanh_f(to_f(s[i])) * e);
}

extern "C" {

void launch_clamped_glu(bool bf16, const GluRows* a, hipStream_t stream) {
  if (bf16)
    clamped_glu_kernel<bf16_t, 8><<<a->blocks(8, 4096), 256, 0, stream>>>(*a);
  else
    clamped_glu_kernel<float, 4><<<a->blocks(4, 4096), 256, 0, stream>>>(*a);
}

void launch_side_gate(bool bf16, float* x_out, const float* x, const void* y, const void* gate,
                      const int64_t* token_ids, const void* table, void* s, int n, int w,
                      int dim, int64_t table_stride, hipStream_t stream) {
  const dim3 grid(n, (dim + 15) / 16);
  if (bf16)
    side_gate_kernel<bf16_t, 8><<<grid, 512, w * 2, stream>>>(
        x_out, x, (const bf16_t*)y, (const bf16_t*)gate, token_ids, (const bf16_t*)table,
        (bf16_t*)s, w, dim, table_stride);
  else
    side_gate_kernel<float, 4><<<grid, 512, w * 4, stream>>>(
        x_out, x, (const float*)y, (const float*)gate, token_ids, (const float*)table, (float*)s, w,
        dim, table_stride);
}

// w a multiple of 8 up to 8192, dim of 8 up to 128
void launch_side_layer(const SideLayerArgs* a, hipStream_t stream) {
  auto launch = [&](auto outputs) {
    constexpr int R = decltype(outputs)::value;
    constexpr int MOST = 8192 * 6 + (16 * R + 48) * 4;
    allow_lds<side_layer_kernel<R>>(MOST);
    side_layer_kernel<R><<<a->n, 1024, a->w * 6 + (16 * R + 48) * 4, stream>>>(*a);
  };
  if (a->dim <= 32) launch(std::integral_constant<int, 2>());
  else if (a->dim <= 64) launch(std::integral_constant<int, 4>());
  else launch(std::integral_constant<int, 8>());
}

void launch_gelu_gate(bool bf16, void* s, const int64_t* token_ids, const void* table,
                      int rows, int dim, int64_t table_stride, hipStream_t stream) {
  const int64_t total = (int64_t)rows * dim;
  const int grid = (int)((total + 255) / 256);
  if (bf16)
    gelu_gate_kernel<bf16_t><<<grid, 256, 0, stream>>>(
        (bf16_t*)s, token_ids, (const bf16_t*)table, dim, total, table_stride);
  else
    gelu_gate_kernel<float><<<grid, 256, 0, stream>>>(
        (float*)s, token_ids, (const float*)table, dim, total, table_stride);
}

}  // extern "C"
