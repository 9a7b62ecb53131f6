// Per-token kernels around latent attention (gfx950): its normed inputs with the
// cache-row write, and the per-head products that absorb the key and value up-projections.
//
// Rotations here pair dimension 2i with 2i+1; cos_sin is [2, P, rot_dim/2] fp32.
#include "common_t.h"
#include "gated_act.h"
#include "latent_attn.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

#define NEG -1e30f

// A wave per token and job.  Job 0: RMS-norm kv[:kv_rank], rotate kv[kv_rank:],
// write the padded cache row [kv_rank -> rank | rot_dim -> row - rank] at its slot.
// Job 1 (low-rank queries): cq = rmsnorm(q) over the first q_rank of its k columns.
// The workgroups past these do the gated unit that reads other columns of the same product, if there is
// one: by itself that is another launch at the cost of one (40 tokens: 4.8 us each, together 4.9).
template <typename T, int V>
__global__ __launch_bounds__(256) void latent_inputs_kernel(
    T* __restrict__ cache, const T* __restrict__ kv, const T* __restrict__ norm_w,
    const int64_t* __restrict__ positions, const int64_t* __restrict__ slots,
    const float* __restrict__ cos_sin, const float eps, const int N,
    const int kv_rank, const int rot_dim, const int rank, const int row,
    const int64_t kv_stride, const int64_t P, T* __restrict__ cq,
    const T* __restrict__ q, const T* __restrict__ q_norm, const int k,
    const int q_rank, const int64_t q_stride, const GluRows glu) {
  const int per_job = (N + 3) / 4, jobs = q ? 2 : 1;
  if ((int)blockIdx.x >= per_job * jobs) {
    const int at = blockIdx.x - per_job * jobs;
    clamped_glu_rows<T, V>(glu, (int64_t)at * 256 + threadIdx.x, (int64_t)(gridDim.x - per_job * jobs) * 256);
    return;
  }
  const bool second = (int)blockIdx.x >= per_job;
  const int n = (blockIdx.x - (second ? per_job : 0)) * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int lane = threadIdx.x & 63;
  if (second) {
    const T* src = q + n * q_stride;
    float ss = 0.f;
    for (int i = lane * V; i < k; i += 64 * V) {
      float t[V];
      load_f<V>(t, src + i);  // columns q_rank.. are zero
#pragma unroll
      for (int j = 0; j < V; ++j) ss += t[j] * t[j];
    }
    const float inv = rsqrtf(wave_sum(ss) / q_rank + eps);
    for (int i = lane * V; i < k; i += 64 * V) {
      float t[V], w[V];
      load_f<V>(t, src + i);
      load_f<V>(w, q_norm + i);
#pragma unroll
      for (int j = 0; j < V; ++j) t[j] *= inv * w[j];
      store_f<V>(cq + (int64_t)n * k + i, t);
    }
    return;
  }
  const T* src = kv + n * kv_stride;
  T* dst = cache + slots[n] * row;
  const int half = rot_dim >> 1;
  const float* ct = cos_sin + positions[n] * half;
  const float* st = ct + P * half;
  for (int i = lane; 2 * i < row - rank; i += 64) {
    float u = 0.f, v = 0.f;
    if (i < half) {
      const float a = to_f(src[kv_rank + 2 * i]), b = to_f(src[kv_rank + 2 * i + 1]);
      u = a * ct[i] - b * st[i];
      v = b * ct[i] + a * st[i];
    }
    const float uv[2] = {u, v};
    store_f<2>(dst + rank + 2 * i, uv);
  }
  float ss = 0.f;
  const bool wide = kv_rank % (64 * V) == 0 &&
                    ((uintptr_t)kv | (uintptr_t)(kv_stride * sizeof(T))) % 16 == 0;
  if (wide) {
    for (int i = lane * V; i < kv_rank; i += 64 * V) {
      float t[V];
      load_f<V>(t, src + i);
#pragma unroll
      for (int j = 0; j < V; ++j) ss += t[j] * t[j];
    }
    const float inv = rsqrtf(wave_sum(ss) / kv_rank + eps);
    for (int i = lane * V; i < kv_rank; i += 64 * V) {
      float t[V], w[V];
      load_f<V>(t, src + i);
      load_f<V>(w, norm_w + i);
#pragma unroll
      for (int j = 0; j < V; ++j) t[j] *= inv * w[j];
      store_f<V>(dst + i, t);
    }
    for (int i = kv_rank + lane; i < rank; i += 64) dst[i] = from_f<T>(0.f);
    return;
  }
  for (int i = lane; i < kv_rank; i += 64) {
    const float f = to_f(src[i]);
    ss += f * f;
  }
  const float inv = rsqrtf(wave_sum(ss) / kv_rank + eps);
  for (int i = lane; i < rank; i += 64)
    dst[i] = from_f<T>(i < kv_rank ? to_f(src[i]) * inv * to_f(norm_w[i]) : 0.f);
}

// out[n, h, :O] = W[h] x[n, h, :K] (* sigmoid(gate[n, h])) on the matrix cores.
// A wave owns 16*OT outputs x 16*TT tokens; both operands are K-contiguous, so the
// fragments load straight from global memory (weights are small enough to stay
// in L2, tokens of one head in L1).  A = weights, B = tokens: a lane ends up
// with 4 consecutive outputs of one token.
template <int OT, int TT>
__global__ __launch_bounds__(256) void head_linear_mfma_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ w, const bf16_t* __restrict__ gate, const int N,
    const int O, const int K, const int64_t x_row, const int x_head,
    const int64_t out_row, const int out_head, const int64_t gate_row) {
  const int h = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const int o0 = (blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6)) * (16 * OT);
  if (o0 >= O) return;
  const int n0 = blockIdx.x * (16 * TT);
  const bf16_t* wp[OT];
  const bf16_t* xp[TT];
#pragma unroll
  for (int i = 0; i < OT; ++i)
    wp[i] = w + ((int64_t)h * O + min(o0 + i * 16 + c, O - 1)) * K + g * 8;
#pragma unroll
  for (int t = 0; t < TT; ++t)
    xp[t] = x + (int64_t)min(n0 + t * 16 + c, N - 1) * x_row + (int64_t)h * x_head + g * 8;
  f32x4_v acc[OT][TT] = {};
#pragma unroll 4
  for (int k = 0; k < K; k += 32) {
    bf16x8_v a[OT], b[TT];
#pragma unroll
    for (int i = 0; i < OT; ++i) a[i] = *(const bf16x8_v*)(wp[i] + k);
#pragma unroll
    for (int t = 0; t < TT; ++t) b[t] = *(const bf16x8_v*)(xp[t] + k);
#pragma unroll
    for (int i = 0; i < OT; ++i)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[t], acc[i][t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    const int n = n0 + t * 16 + c;
    if (n >= N) continue;
    const float s = gate ? sigmoid_f(bf2f(gate[n * gate_row + h])) : 1.f;
    bf16_t* dst = out + n * out_row + (int64_t)h * out_head;
#pragma unroll
    for (int i = 0; i < OT; ++i) {
      const int o = o0 + i * 16 + g * 4;  // O is a multiple of 32
      if (o >= O) continue;
      const float v[4] = {acc[i][t][0] * s, acc[i][t][1] * s, acc[i][t][2] * s,
                          acc[i][t][3] * s};
      store_f<4>(dst + o, v);
    }
  }
}

// out[n, h, :O] = W[h] x[n, h, :K] (* sigmoid(gate[n, h])) of rows x that are still in n_split parts (SplitOut):
// a workgroup merges its T <= 16 tokens of one head into LDS, rounded as a merge by itself rounds them, and its 8
// waves take 16 outputs each.  Everything is on its way from the start (a wave's first weights, the parts,
// their sums): what is left is one latency and the reads, 128 KB of weights and T n_split 2 KB at a rank of 512.
// Heads are neighbours in the grid, so that an XCD reads its heads' weights alone.
// 40 tokens of 16 heads of rank 512 in 6 parts, 128 outputs: 8.0 us, before, merged (4.9) and multiplied (9.2), 14.1
// and a gap between launches; attention and this together 40 x 3000 47.4 -> 42.9, 250 x 2000 in 2 parts
// 116.3 -> 112.4, one of 300 keys 19.3 -> 16.5.
template <int KS>  // K / 32
__global__ __launch_bounds__(512) void merge_head_linear_kernel(const MergedHeads a) {
  constexpr int K = KS * 32, BATCH = 8;
  __shared__ bf16_t rows[16][K + 8];
  __shared__ float weight[16][64];
  __shared__ int live[16];
  const int h = blockIdx.x, n0 = blockIdx.y * a.T, tokens = min(a.T, a.N - n0);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int64_t n_rows = (int64_t)a.N * a.H;
  const float* const part = a.part + ((int64_t)n0 * a.H + h) * K;

  float4 v[BATCH];
  auto load_parts = [&](int t, int k, int from, int some) {
#pragma unroll
    for (int s = 0; s < BATCH; ++s)
      v[s] = *(const float4*)(part + (min(from + s, some - 1) * n_rows + (int64_t)t * a.H) * K + k);
  };
  bf16x8_v w[KS];
  auto load_weights = [&](int o) {
    const bf16_t* src = (const bf16_t*)a.w + ((int64_t)h * a.O + min(o + c, a.O - 1)) * K + g * 8;
#pragma unroll
    for (int k = 0; k < KS; ++k) w[k] = *(const bf16x8_v*)(src + k * 32);
  };
  const int at0 = threadIdx.x * 4;
  load_parts(min(at0 / K, tokens - 1), at0 % K, 0, a.usual);
  load_weights(wid * 16);

  for (int t = wid; t < tokens; t += 8) {
    const float2 ml = lane < a.n_split ? a.part_ml[lane * n_rows + (int64_t)(n0 + t) * a.H + h] : float2{NEG, -1.f};
    const int some = __popcll(__ballot(ml.y >= 0.f));
    const float m = wave_max(ml.x);
    const float e = ml.y > 0.f ? __builtin_amdgcn_exp2f(ml.x - m) : 0.f;
    const float l = wave_sum(e * fmaxf(ml.y, 0.f));
    weight[t][lane] = l > 0.f ? e / l : 0.f;
    if (lane == 0) live[t] = some;
  }
  __syncthreads();
  for (int at = at0; at < 16 * K; at += 2048) {
    const int t = at / K, k = at % K;
    float acc[4] = {};
    if (t < tokens) {
      for (int from = 0; from < live[t]; from += BATCH) {
        if (at != at0 || from || live[t] > a.usual) load_parts(t, k, from, live[t]);
#pragma unroll
        for (int s = 0; s < BATCH; ++s)
          if (from + s < live[t]) {
            const float p = weight[t][from + s];
            acc[0] += p * v[s].x;
            acc[1] += p * v[s].y;
            acc[2] += p * v[s].z;
            acc[3] += p * v[s].w;
          }
      }
    }
    store_f<4>(&rows[t][k], acc);
  }
  __syncthreads();
  const bool mine = c < tokens;
  const int64_t n = n0 + min(c, tokens - 1);
  const float s = a.gate ? sigmoid_f(bf2f(((const bf16_t*)a.gate)[n * a.gate_row + h])) : 1.f;
  for (int o = wid * 16; o < a.O; o += 128) {
    if (o != wid * 16) load_weights(o);
    f32x4_v acc = {};
#pragma unroll
    for (int k = 0; k < KS; ++k)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k], *(const bf16x8_v*)&rows[c][k * 32 + g * 8], acc, 0, 0, 0);
    const float y[4] = {acc[0] * s, acc[1] * s, acc[2] * s, acc[3] * s};
    if (mine) store_f<4>((bf16_t*)a.out + n * a.out_row + (int64_t)h * a.out_head + o + g * 4, y);
  }
}

// fp32 twin: a thread per output, 4 tokens per block in flight.
__global__ __launch_bounds__(256) void head_linear_f32_kernel(
    float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,
    const float* __restrict__ gate, const int N, const int O, const int K,
    const int64_t x_row, const int x_head, const int64_t out_row,
    const int out_head, const int64_t gate_row) {
  const int h = blockIdx.z;
  const int o = blockIdx.y * 64 + (threadIdx.x & 63);
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (o >= O || n >= N) return;
  const float* wr = w + ((int64_t)h * O + o) * K;
  const float* xr = x + n * x_row + (int64_t)h * x_head;
  float acc = 0.f;
  for (int k = 0; k < K; k += 4) {
    float a[4], b[4];
    load_f<4>(a, wr + k);
    load_f<4>(b, xr + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc += a[j] * b[j];
  }
  if (gate) acc *= sigmoid_f(gate[n * gate_row + h]);
  out[n * out_row + (int64_t)h * out_head + o] = acc;
}

extern "C" {

void launch_latent_inputs(bool bf16, void* cache, const void* kv, const void* norm_w,
                          const int64_t* positions, const int64_t* slots,
                          const float* cos_sin, float eps, int N, int kv_rank, int rot_dim,
                          int rank, int row, int64_t kv_stride, int64_t P, void* cq,
                          const void* q, const void* q_norm, int k, int q_rank,
                          int64_t q_stride, const GluRows* glu, hipStream_t stream) {
  const int grid = (N + 3) / 4 * (q ? 2 : 1) + (glu ? glu->blocks(bf16 ? 8 : 4, 4096) : 0);
  const GluRows rows = glu ? *glu : GluRows{};
  if (bf16)
    latent_inputs_kernel<bf16_t, 8><<<grid, 256, 0, stream>>>(
        (bf16_t*)cache, (const bf16_t*)kv, (const bf16_t*)norm_w, positions, slots,
        cos_sin, eps, N, kv_rank, rot_dim, rank, row, kv_stride, P, (bf16_t*)cq,
        (const bf16_t*)q, (const bf16_t*)q_norm, k, q_rank, q_stride, rows);
  else
    latent_inputs_kernel<float, 4><<<grid, 256, 0, stream>>>(
        (float*)cache, (const float*)kv, (const float*)norm_w, positions, slots, cos_sin,
        eps, N, kv_rank, rot_dim, rank, row, kv_stride, P, (float*)cq, (const float*)q,
        (const float*)q_norm, k, q_rank, q_stride, rows);
}

// K one of 64 128 256 384 512, O a multiple of 32, n_split at most 64
void launch_merge_head_linear(const MergedHeads* a, int K, hipStream_t stream) {
  MergedHeads m = *a;
  // tokens of a workgroup: as few as leave one to a CU, since each of them reads the head's weights
  m.T = (int64_t)m.N * m.H <= 1024 ? 4 : (int64_t)m.N * m.H <= 2048 ? 8 : 16;
  const dim3 grid(m.H, (m.N + m.T - 1) / m.T);
  auto k = K == 64    ? merge_head_linear_kernel<2>
           : K == 128 ? merge_head_linear_kernel<4>
           : K == 256 ? merge_head_linear_kernel<8>
           : K == 384 ? merge_head_linear_kernel<12>
                      : merge_head_linear_kernel<16>;
  k<<<grid, 512, 0, stream>>>(m);
}

void launch_head_linear(bool bf16, void* out, const void* x, const void* w,
                        const void* gate, int N, int H, int O, int K, int64_t x_row,
                        int x_head, int64_t out_row, int out_head, int64_t gate_row,
                        hipStream_t stream) {
  if (!bf16) {
    dim3 grid((N + 3) / 4, (O + 63) / 64, H);
    head_linear_f32_kernel<<<grid, 256, 0, stream>>>(
        (float*)out, (const float*)x, (const float*)w, (const float*)gate, N, O, K,
        x_row, x_head, out_row, out_head, gate_row);
    return;
  }
  // few tokens: small wave tiles, so that enough waves hide the load latency
  const int tt = N > 2048 ? 4 : N > 256 ? 2 : 1;
  const int ot = tt == 1 ? 2 : 4;
  const int tiles = (O + 16 * ot - 1) / (16 * ot);
  const int waves = tiles < 4 ? tiles : 4;
  dim3 grid((N + 16 * tt - 1) / (16 * tt), (tiles + waves - 1) / waves, H);
  auto k = tt == 4 ? head_linear_mfma_kernel<4, 4>
                   : tt == 2 ? head_linear_mfma_kernel<4, 2> : head_linear_mfma_kernel<2, 1>;
  k<<<grid, 64 * waves, 0, stream>>>(
      (bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)gate, N, O, K,
      x_row, x_head, out_row, out_head, gate_row);
}

}  // extern "C"
