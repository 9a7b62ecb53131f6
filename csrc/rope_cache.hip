// Fused rotary embedding + paged-KV scatter (gfx950).
//
// One kernel applies rotate-half RoPE to Q and K in place and scatters the
// post-rope K and raw V of every token into the paged cache at its flat
// slot — one pass over the QKV projection output instead of the three the
// unfused form costs (rope q, rope k, cache write).
//
// Layouts: q [N, Hq, D], k/v [N, Hkv, D] bf16 contiguous; cache
// [num_blocks, block_size, Hkv, D] viewed flat as [slots, Hkv, D];
// cos_sin [2, P, D/2] fp32.  D = head_dim (128 for the model family).
#include "common.h"

__global__ void rope_cache_kernel(
    bf16_t* __restrict__ q,            // [N, Hq, D], token stride q_stride
    bf16_t* __restrict__ k,            // [N, Hkv, D], token stride kv_stride
    const bf16_t* __restrict__ v,      // [N, Hkv, D], token stride kv_stride
    bf16_t* __restrict__ k_cache,      // [slots, Hkv, D]
    bf16_t* __restrict__ v_cache,
    const int64_t* __restrict__ positions,     // [N]
    const int64_t* __restrict__ slot_mapping,  // [N]
    const float* __restrict__ cos_sin,         // [2, P, D/2]
    const int Hq, const int Hkv, const int D, const int64_t P,
    const int64_t q_stride, const int64_t kv_stride) {
  const int token = blockIdx.x;
  const int64_t pos = positions[token];
  const int64_t slot = slot_mapping[token];
  const int d2 = D >> 1;
  const float* cos_t = cos_sin + pos * d2;
  const float* sin_t = cos_sin + (P + pos) * d2;

  const int wid = threadIdx.x >> 6;      // wave id
  const int lane = threadIdx.x & 63;
  const int nw = blockDim.x >> 6;
  const int per_lane = d2 / WAVE;        // rotate pairs per lane (D=128 → 1)

  // Q heads: rope in place
  for (int hq = wid; hq < Hq; hq += nw) {
    bf16_t* qh = q + (int64_t)token * q_stride + (int64_t)hq * D;
#pragma unroll
    for (int r = 0; r < 4; ++r) {        // supports D up to 512
      if (r >= per_lane) break;
      const int i = lane + (r << 6);
      const float c = cos_t[i], s = sin_t[i];
      const float x1 = bf2f(qh[i]), x2 = bf2f(qh[i + d2]);
      qh[i] = f2bf(x1 * c - x2 * s);
      qh[i + d2] = f2bf(x2 * c + x1 * s);
    }
  }
  // K heads: rope in place + cache scatter; V heads: cache scatter
  for (int hk = wid; hk < Hkv; hk += nw) {
    bf16_t* kh = k + (int64_t)token * kv_stride + (int64_t)hk * D;
    const bf16_t* vh = v + (int64_t)token * kv_stride + (int64_t)hk * D;
    bf16_t* kc = k_cache + (slot * Hkv + hk) * D;
    bf16_t* vc = v_cache + (slot * Hkv + hk) * D;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r >= per_lane) break;
      const int i = lane + (r << 6);
      const float c = cos_t[i], s = sin_t[i];
      const float x1 = bf2f(kh[i]), x2 = bf2f(kh[i + d2]);
      const bf16_t k1 = f2bf(x1 * c - x2 * s), k2 = f2bf(x2 * c + x1 * s);
      kh[i] = k1;
      kh[i + d2] = k2;
      kc[i] = k1;
      kc[i + d2] = k2;
      vc[i] = vh[i];
      vc[i + d2] = vh[i + d2];
    }
  }
}

// The same in units of 8 pairs, 256 of a step's units a workgroup, so that few tokens fill more
// than as many CUs and no wave takes a token's heads in turn: heads of a multiple of 16, rows
// of 16-byte units.  13 tokens of 96 heads (queries, keys, values) 10.5 to 4.8 us, 61 of 48 7.4
// to 4.8, 15675 of 48 84 to 71.
// With PARTS the projection is fp32 [n_parts, N, (Hq + 2 Hkv) D], sums over parts of the inner
// dimension (linear.hip) that are added up in their order and rounded, as their own pass would
// do; queries go to q, keys and values to their slots alone.
template <bool PARTS>
__global__ __launch_bounds__(256) void rope_cache_units_kernel(
    bf16_t* __restrict__ q, bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache,
    const int64_t* __restrict__ positions, const int64_t* __restrict__ slot_mapping,
    const float* __restrict__ cos_sin, const int N, const int Hq, const int Hkv, const int D,
    const int64_t P, const int64_t q_stride, const int64_t kv_stride,
    const float* __restrict__ parts, const int n_parts) {
  const int d2 = D >> 1, per = d2 >> 3, heads = Hq + 2 * Hkv;
  const int64_t unit = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = unit / per;  // of heads
  const int i = (int)(unit - row * per) * 8;
  const int64_t token = row / heads;
  if (token >= N) return;
  const int head = (int)(row - token * heads), kv = head < Hq + Hkv ? head - Hq : head - Hq - Hkv;
  const bool is_q = head < Hq, is_v = head >= Hq + Hkv;
  bf16_t* const at = is_q ? q + token * q_stride + (int64_t)head * D + i
                          : (bf16_t*)(is_v ? v : k) + token * kv_stride + (int64_t)kv * D + i;
  const int64_t slot = is_q ? 0 : slot_mapping[token];
  BF16x8 a, b;
  if (PARTS) {
    const float* from = parts + (token * heads + head) * D + i;
    float y[16] = {};
#pragma unroll 4
    for (int p = 0; p < n_parts; ++p, from += (int64_t)N * heads * D) {
#pragma unroll
      for (int e = 0; e < 16; e += 4) {
        const float4 c = *(const float4*)(from + (e < 8 ? e : d2 + e - 8));
        y[e] += c.x; y[e + 1] += c.y; y[e + 2] += c.z; y[e + 3] += c.w;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a.h[e] = f2bf(y[e]);
      b.h[e] = f2bf(y[8 + e]);
    }
  } else {
    a = *(const BF16x8*)at;
    b = *(const BF16x8*)(at + d2);
  }
  if (!is_v) {
    const int64_t pos = positions[token];
    const float* cos_t = cos_sin + pos * d2 + i;
    const float* sin_t = cos_sin + (P + pos) * d2 + i;
    float c[8], s[8];
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      *(float4*)(c + e) = *(const float4*)(cos_t + e);
      *(float4*)(s + e) = *(const float4*)(sin_t + e);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x1 = bf2f(a.h[e]), x2 = bf2f(b.h[e]);
      a.h[e] = f2bf(x1 * c[e] - x2 * s[e]);
      b.h[e] = f2bf(x2 * c[e] + x1 * s[e]);
    }
    if (is_q || !PARTS) {
      *(BF16x8*)at = a;
      *(BF16x8*)(at + d2) = b;
    }
  }
  if (!is_q) {
    bf16_t* const to = (is_v ? v_cache : k_cache) + (slot * Hkv + kv) * D + i;
    *(BF16x8*)to = a;
    *(BF16x8*)(to + d2) = b;
  }
}

extern "C" void launch_rope_cache_units(void* q, void* k, const void* v, void* k_cache,
                                        void* v_cache, const int64_t* positions,
                                        const int64_t* slot_mapping, const float* cos_sin, int N,
                                        int Hq, int Hkv, int D, int64_t P, int64_t q_stride,
                                        int64_t kv_stride, const float* parts, int n_parts,
                                        hipStream_t stream) {
  const int64_t units = (int64_t)N * (Hq + 2 * Hkv) * (D / 16);
  auto kernel = parts ? rope_cache_units_kernel<true> : rope_cache_units_kernel<false>;
  kernel<<<dim3((units + 255) / 256), 256, 0, stream>>>(
      (bf16_t*)q, (bf16_t*)k, (const bf16_t*)v, (bf16_t*)k_cache, (bf16_t*)v_cache, positions,
      slot_mapping, cos_sin, N, Hq, Hkv, D, P, q_stride, kv_stride, parts, n_parts);
}

extern "C" void launch_rope_cache(void* q, void* k, const void* v,
                                  void* k_cache, void* v_cache,
                                  const int64_t* positions,
                                  const int64_t* slot_mapping,
                                  const float* cos_sin, int N, int Hq,
                                  int Hkv, int D, int64_t P,
                                  int64_t q_stride, int64_t kv_stride,
                                  hipStream_t stream) {
  dim3 grid(N), block(256);
  hipLaunchKernelGGL(rope_cache_kernel, grid, block, 0, stream, (bf16_t*)q,
                     (bf16_t*)k, (const bf16_t*)v, (bf16_t*)k_cache,
                     (bf16_t*)v_cache, positions, slot_mapping, cos_sin, Hq,
                     Hkv, D, P, q_stride, kv_stride);
}
