// Mixture of experts (gfx950): routing, grouping by expert, and the experts' products
// for few rows per expert and for fp32.  experts_gemm.hip has the product for many.
//
// Nothing here depends on the routing but memory contents: grids come from host values,
// so decode steps can be captured.
#include "experts.h"
#include "gated_act.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

#define ROUTE_T 16  // tokens per workgroup
#define ROUTE_WAVES 4     // of a workgroup that has a part of K
#define ROUTE_MOST 1024
#define AHEAD 8      // turns whose ids are loaded together

// The wave picks the ``top`` largest of logits[0 .. E) (overwritten), the lower index
// among equals, and their weights: scale times their softmax or, with ``scores``, times
// the chosen scores over their sum.
static DEV void choose(float* logits, const float* scores, int E, int top, float scale, int* ids,
                       float* weights) {
  const int lane = threadIdx.x & 63;
  float mine = -INFINITY, first = 0.f;
  int my_id = 0;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 1 << 30;
    for (int e = lane; e < E; e += 64)
      if (logits[e] > best) {
        best = logits[e];
        at = e;
      }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float v = __shfl_xor(best, off, 64);
      const int i = __shfl_xor(at, off, 64);
      if (v > best || (v == best && i < at)) {
        best = v;
        at = i;
      }
    }
    at = min(at, E - 1);  // whatever the logits are, an id stays an id
    if (j == 0) first = best;
    if (lane == j) {
      mine = scores ? scores[at] : best;
      my_id = at;
    }
    if (lane == (at & 63)) logits[at] = -INFINITY;
  }
  const float w = lane >= top ? 0.f : scores ? mine : expf(mine - first);
  const float sum = wave_sum(w) + (scores ? 1e-20f : 0.f);
  if (lane < top) {
    ids[lane] = my_id;
    weights[lane] = scale * w / sum;
  }
}

// 16 tokens a workgroup: its waves split K in blocks of 64, partial logits meet in LDS.
// NF fragments of 16 experts at a time.
// Dynamic LDS: [waves][16][E16] floats, E16 = E rounded up to 16.
// A CU takes about 25 GB/s from memory, so the weights of 32 experts of 4096 take one 10 us,
// and few tokens leave the others idle.  With ``sums`` [parts of K][N][E16] the workgroups of
// grid row y take part y of K, and route_sums_kernel chooses: 48 tokens, 32 experts of 4096
// 18.4 to 11.1 us for both launches.
template <int NF>
__global__ __launch_bounds__(1024) void route_mfma_kernel(
    int* __restrict__ ids, float* __restrict__ weights, const bf16_t* __restrict__ h,
    const bf16_t* __restrict__ w, const float* __restrict__ bias, const int N, const int E,
    const int K, const int top, const int64_t h_stride, const bool sigmoid, const float scale,
    float* __restrict__ sums) {
  extern __shared__ float part[];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int blocks = gridDim.y * waves, block = blockIdx.y * waves + wid;
  const int E16 = (E + 15) & ~15, logits = ROUTE_T * E16;
  const int n0 = blockIdx.x * ROUTE_T;
  const bf16_t* hp = h + (int64_t)min(n0 + c, N - 1) * h_stride + g * 8;
  float* mine = part + (int64_t)wid * logits;
  for (int e0 = 0; e0 < E16; e0 += 16 * NF) {
    const bf16_t* wp[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i)
      wp[i] = w + (int64_t)min(e0 + i * 16 + c, E - 1) * K + g * 8;
    f32x4_v acc[NF] = {};
#pragma unroll 4
    for (int k = block * 64; k < K; k += blocks * 64) {
#pragma unroll
      for (int s = 0; s < 64; s += 32) {
        const bf16x8_v b = *(const bf16x8_v*)(hp + k + s);
#pragma unroll
        for (int i = 0; i < NF; ++i) {
          const bf16x8_v f = *(const bf16x8_v*)(wp[i] + k + s);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, b, acc[i], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const int e = e0 + i * 16 + g * 4;
      if (e < E16) *(f32x4_v*)(mine + c * E16 + e) = acc[i];
    }
  }
  __syncthreads();
  // the first wave's part becomes the logits, the second's the scores
  for (int i = threadIdx.x; i < logits; i += blockDim.x) {
    const int e = i % E16;
    float z = 0.f;
    for (int p = 0; p < waves; ++p) z += part[(int64_t)p * logits + i];
    if (sums) {
      const int n = n0 + i / E16;
      if (n < N) sums[((int64_t)blockIdx.y * N + n) * E16 + e] = z;
      continue;
    }
    if (sigmoid) part[logits + i] = z = 1.f / (1.f + expf(-z));
    part[i] = e < E ? z + (bias ? bias[e] : 0.f) : -INFINITY;
  }
  if (sums) return;
  __syncthreads();
  for (int t = wid; t < min(ROUTE_T, N - n0); t += waves)
    choose(part + t * E16, sigmoid ? part + logits + t * E16 : nullptr, E, top, scale,
           ids + (int64_t)(n0 + t) * top, weights + (int64_t)(n0 + t) * top);
}

// The logits from their parts, in order; a wave a token, at most 128 experts.
__global__ __launch_bounds__(64) void route_sums_kernel(
    int* __restrict__ ids, float* __restrict__ weights, const float* __restrict__ sums,
    const float* __restrict__ bias, const int N, const int E, const int parts, const int top,
    const bool sigmoid, const float scale) {
  __shared__ float logits[128], scores[128];
  const int E16 = (E + 15) & ~15;
  const int64_t n = blockIdx.x;
  for (int e = threadIdx.x; e < E; e += 64) {
    float z = 0.f;
#pragma unroll 16
    for (int p = 0; p < parts; ++p) z += sums[((int64_t)p * N + n) * E16 + e];
    if (sigmoid) scores[e] = z = 1.f / (1.f + expf(-z));
    logits[e] = z + (bias ? bias[e] : 0.f);
  }
  __syncthreads();
  choose(logits, sigmoid ? scores : nullptr, E, top, scale, ids + n * top, weights + n * top);
}

// Any dtype: a workgroup per token, a wave per expert in turn.
template <typename T>
__global__ __launch_bounds__(256) void route_plain_kernel(
    int* __restrict__ ids, float* __restrict__ weights, const T* __restrict__ h,
    const T* __restrict__ w, const float* __restrict__ bias, const int E, const int K,
    const int top, const int64_t h_stride, const bool sigmoid, const float scale) {
  extern __shared__ float part[];  // [2][E]
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t n = blockIdx.x;
  for (int e = wid; e < E; e += 4) {
    float z = 0.f;
    for (int k = lane; k < K; k += 64) z += to_f(h[n * h_stride + k]) * to_f(w[(int64_t)e * K + k]);
    z = wave_sum(z);
    if (sigmoid) z = 1.f / (1.f + expf(-z));
    if (lane == 0) {
      part[E + e] = z;
      part[e] = z + (bias ? bias[e] : 0.f);
    }
  }
  __syncthreads();
  if (wid == 0)
    choose(part, sigmoid ? part + E : nullptr, E, top, scale, ids + n * top, weights + n * top);
}

// lanes of the wave whose id (``bits`` bits) equals this lane's
static DEV uint64_t same_id(int id, int bits) {
  uint64_t m = ~0ull;
  for (int b = 0; b < bits; ++b) {
    const uint64_t set = __ballot((id >> b) & 1);
    m &= (id >> b) & 1 ? set : ~set;
  }
  return m;
}

// Group the entries by expert, in their order: a counting sort.  Every workgroup counts all
// entries (atomics in LDS), its waves their own runs of its share as well, which they then
// place; the last one lists the tiles.  One workgroup for all, whose waves placed 1 / 16 each,
// took 33.6 us for 16372 entries of 32 experts with the tiles (now 14.4), 8.9 for 192 (now 7.1).
// Dynamic LDS: [18][E] ints.
template <bool TILED>
__global__ __launch_bounds__(1024) void group_kernel(
    int* __restrict__ perm, int* __restrict__ offsets, int* __restrict__ tile_expert,
    int* __restrict__ tile_row, const int* __restrict__ ids, const int n, const int E) {
  extern __shared__ int counts[];
  __shared__ int step_tiles[EXPERT_TILE / 32];
  int* total = counts + 16 * E;
  int* earlier = total + E;  // in the shares before this one
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int bits = 32 - __clz(E);  // E itself marks lanes past the end
  const int shares = gridDim.x - 1, per = ((n + shares - 1) / shares + 1023) / 1024 * 64;  // a wave's
  const bool lists = blockIdx.x == shares;
  const int share = blockIdx.x * per * 16;
  for (int i = threadIdx.x; i < 18 * E; i += 1024) counts[i] = 0;
  __syncthreads();
  auto turns = [&](int i0, int i1, int step, auto&& turn) {  // with the ids loaded ahead
    for (int i = i0; i < i1; i += step * AHEAD) {
      int id[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        const int at = i + j * step;
        id[j] = at < i1 ? ids[at] : E;
      }
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) turn(i + j * step, id[j]);
    }
  };
  turns(threadIdx.x, n, 1024, [&](int at, int id) {
    if (id >= E) return;
    atomicAdd(&total[id], 1);
    if (at < share) atomicAdd(&earlier[id], 1);
  });
  const int i0 = lists ? n : share + wid * per, i1 = min(n, i0 + per);
  int* mine = counts + wid * E;
  turns(i0 + lane, i1, 64, [&](int, int id) {
    if (id < E) atomicAdd(&mine[id], 1);
  });
  __syncthreads();
  if (!lists)
    for (int e = threadIdx.x; e < E; e += 1024) {
      int run = earlier[e];
      for (int w = 0; w < 16; ++w) {
        const int t = counts[w * E + e];
        counts[w * E + e] = run;
        run += t;
      }
    }
  auto before = [&](int v, int& sum) {  // the lanes before this one's; the wave's sum
    int s = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int w = __shfl_up(s, off, 64);
      if (lane >= off) s += w;
    }
    sum = __shfl(s, 63, 64);
    return s - v;
  };
  if (lists) {  // first rows of the experts and their tiles
    // an expert's tiles have the same height
    auto tiles_of = [&](int c, int& high) {
      const int t = TILED ? (c + EXPERT_TILE - 1) / EXPERT_TILE : 0;
      high = t > 0 ? (c + t - 1) / t : 0;
      return t;
    };
    // the highest tiles first, by steps of 32 rows, a wave each: workgroups that end early then
    // fill up with the lower ones
    const int steps = TILED ? EXPERT_TILE / 32 : 0;
    const int step = steps - wid;  // of rows
    int tile = 0;
    auto list = [&](bool count) {
      int row = 0, sum;
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane, c = e < E ? total[e] : 0;
        int high;
        int t = tiles_of(c, high);
        if ((high + 31) / 32 != step) t = 0;
        const int first = row + before(c, sum);
        row += sum;
        const int at = tile + before(t, sum);
        tile += sum;
        for (int j = 0; j < t && !count; ++j) {
          tile_expert[at + j] = e;
          tile_row[at + j] = first + j * high;
        }
      }
    };
    if (step > 0) {
      list(true);
      if (lane == 0) step_tiles[wid] = tile;
    }
    __syncthreads();
    if (step > 0) {
      tile = 0;
      for (int w = 0; w < wid; ++w) tile += step_tiles[w];
      list(false);
    }
    if (wid == 15) {
      int row = 0, sum;
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        const int first = row + before(e < E ? total[e] : 0, sum);
        row += sum;
        if (e < E) offsets[e] = first;
      }
      if (lane == 0) {
        offsets[E] = row;
        tile = 0;
        for (int w = 0; w < steps; ++w) tile += step_tiles[w];
        offsets[E + 1] = tile;
      }
    }
    return;
  }
  if (wid == 0) {
    int row = 0, sum;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane;
      const int first = row + before(e < E ? total[e] : 0, sum);
      row += sum;
      if (e < E) total[e] = first;
    }
  }
  __syncthreads();
  turns(i0 + lane, i1, 64, [&](int at, int id) {
    const uint64_t m = same_id(id, bits);
    const int leader = __builtin_ctzll(m);
    int base = 0;
    if (id < E && lane == leader) {
      base = mine[id];
      mine[id] = base + __popcll(m);
    }
    asm volatile("" ::: "memory");
    base = __shfl(base, leader, 64);
    if (id < E) perm[total[id] + base + __popcll(m & ((1ull << lane) - 1))] = at;
  });
}

// Four outputs of a row from its sums, with GLU of the gates y and ups u
template <bool GLU>
static DEV void store_outputs(const ExpertsArgs& a, int64_t row, int o, f32x4_v v, f32x4_v u) {
  float y[4] = {v[0], v[1], v[2], v[3]};
  if (GLU) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // through the model's precision, as a GEMM stores it
      const float gate = to_f(from_f<bf16_t>(y[k])), up = to_f(from_f<bf16_t>(u[k]));
      y[k] = clamped_glu_f(gate, up, a.limit, a.alpha, a.offset, a.cubic);
    }
  }
  bf16_t* dst = (bf16_t*)a.out + row * a.O + o;
  if (a.O % 4 == 0)
    store_f<4>(dst, y);
  else
    for (int k = 0; k < 4 && o + k < a.O; ++k) dst[k] = from_f<bf16_t>(y[k]);
}

// Few rows per expert: bound by the weights.  grid (outputs / 16 or 32, E); the 4 waves
// of a workgroup split K in blocks of 64 and meet in LDS.  Two tiles of 16 rows of weights: gate
// and up of the same 16 outputs, or 32 outputs.  A load has 8 rows of a whole line (64 of K), past
// the caches: a model's other layers have come between.  The upper 8 rows and columns of a product
// have the line's other half, and of its results those count whose row and column have the same
// half; 8 TT tokens at a time.  Both products with routing, weights from memory, us, by loads of 16
// rows of half a line through the caches, and so: 32 experts of 4096 x 2560, 4 a token, 2 tokens 129
// and 105, 8 252 and 225, 48 374 and 334, 95 413 and 376; 16 of 2048 x 1536 1 token 42 and 42, 4 66 and
// 59, 8 75 and 70, 16 78.5 and 74, 32 79 and 77.  Weights that are still in the caches, as in a loop
// over one layer, are no slower so but for 1 and 2 tokens of the smaller ones (38 and 42, 47 and 53).
template <bool GLU, int TT>
__global__ __launch_bounds__(256) void experts_small_kernel(const ExpertsArgs a) {
  __shared__ f32x4_v red[4][2][2][TT][2][16];  // wave, tile, 8 rows, tokens, half, (4 rows, token)
  const int e = blockIdx.y;
  const int row0 = a.offsets[e], rows = a.offsets[e + 1] - row0;
  if (rows == 0) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane & 7, half = lane >> 3 & 1, j = lane >> 4, in = half * 32 + j * 8;
  const int o0 = blockIdx.x * (GLU ? 16 : 32);
  const bf16_t* w = (const bf16_t*)a.w + (int64_t)e * (GLU ? 2 : 1) * a.O * a.K + in;
  const bf16_t* wp[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int o = GLU ? o0 + p * 8 + c + i * a.O : min(o0 + i * 16 + p * 8 + c, a.O - 1);
      wp[i][p] = w + (int64_t)o * a.K;
    }
  for (int r0 = 0; r0 < rows; r0 += 8 * TT) {
    const bf16_t* xp[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const int r = row0 + min(r0 + t * 8 + c, rows - 1);
      xp[t] = (const bf16_t*)a.x + (int64_t)(GLU ? a.perm[r] / a.top : r) * a.x_stride + in;
    }
    f32x4_v acc[2][2][TT] = {};
#pragma unroll 2
    for (int k = wid * 64; k < a.K; k += 256) {
      bf16x8_v f[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          f[i][p] = __builtin_nontemporal_load((const bf16x8_v*)(wp[i][p] + k));
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const bf16x8_v b = *(const bf16x8_v*)(xp[t] + k);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int p = 0; p < 2; ++p)
            acc[i][p][t] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i][p], b, acc[i][p][t], 0, 0, 0);
      }
    }
    if (r0) __syncthreads();
    if (half == j >> 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int t = 0; t < TT; ++t) red[wid][i][p][t][half][(j & 1) * 8 + c] = acc[i][p][t];
    }
    __syncthreads();
    // a thread sums 4 outputs of one row
    for (int n = threadIdx.x; n < (GLU ? 1 : 2) * 2 * TT * 16; n += 256) {
      const int l = n & 15, t = (n >> 4) % TT, p = (n >> 4) / TT & 1, i = (n >> 5) / TT;
      const int r = r0 + t * 8 + (l & 7), o = o0 + i * 16 + p * 8 + (l >> 3) * 4;
      if (r >= rows || o >= a.O) continue;
      auto sum = [&](int i) {
        f32x4_v v = {};
#pragma unroll
        for (int x = 0; x < 4; ++x) v += red[x][i][p][t][0][l] + red[x][i][p][t][1][l];
        return v;
      };
      store_outputs<GLU>(a, GLU ? row0 + r : a.perm[row0 + r], o, sum(i), sum(1));
    }
  }
}

// fp32: a thread per output; rows are entries in both products, nothing is grouped.
template <bool GLU>
__global__ __launch_bounds__(256) void experts_f32_kernel(const ExpertsArgs a) {
  const int o = blockIdx.y * 64 + (threadIdx.x & 63);
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (o >= a.O || i >= a.entries) return;
  const float* w = (const float*)a.w + ((int64_t)a.ids[i] * (GLU ? 2 : 1) * a.O + o) * a.K;
  const float* x = (const float*)a.x + (int64_t)(GLU ? i / a.top : i) * a.x_stride;
  float g = 0.f, u = 0.f;
  for (int k = 0; k < a.K; k += 4) {
    float xv[4], wv[4];
    load_f<4>(xv, x + k);
    load_f<4>(wv, w + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) g += xv[j] * wv[j];
    if (GLU) {
      load_f<4>(wv, w + (int64_t)a.O * a.K + k);
#pragma unroll
      for (int j = 0; j < 4; ++j) u += xv[j] * wv[j];
    }
  }
  ((float*)a.out)[(int64_t)i * a.O + o] =
      GLU ? clamped_glu_f(g, u, a.limit, a.alpha, a.offset, a.cubic) : g;
}

extern "C" {

// Parts of K for few tokens: a block of 64 a wave, and no more workgroups than CUs; from
// ROUTE_MOST tokens on the CUs are busy as it is
int moe_route_parts(bool bf16, int N, int E, int K) {
  const int tiles = (N + ROUTE_T - 1) / ROUTE_T;
  if (!bf16 || E > 128 || N >= ROUTE_MOST) return 1;
  return max(1, min(256 / tiles, K / (64 * ROUTE_WAVES)));
}

void launch_moe_route(bool bf16, int* ids, float* weights, const void* h, const void* w,
                      const float* bias, int N, int E, int K, int top, int64_t h_stride,
                      bool sigmoid, float scale, float* sums, int parts, hipStream_t stream) {
  const int E16 = (E + 15) & ~15;
  if (bf16 && E <= 128) {  // at most 64 KiB of partial logits
    // few workgroups: more waves share the weights' latency
    const int waves = parts > 1 ? ROUTE_WAVES : N <= 4096 && E16 <= 64 ? 16 : 8;
    auto k = E16 <= 16   ? route_mfma_kernel<1>
             : E16 <= 32 ? route_mfma_kernel<2>
                         : route_mfma_kernel<4>;
    k<<<dim3((N + ROUTE_T - 1) / ROUTE_T, parts), 64 * waves, waves * ROUTE_T * E16 * 4, stream>>>(
        ids, weights, (const bf16_t*)h, (const bf16_t*)w, bias, N, E, K, top, h_stride, sigmoid,
        scale, parts > 1 ? sums : nullptr);
    if (parts > 1)
      route_sums_kernel<<<N, 64, 0, stream>>>(ids, weights, sums, bias, N, E, parts, top, sigmoid,
                                              scale);
  } else if (bf16) {
    route_plain_kernel<bf16_t><<<N, 256, E * 8, stream>>>(
        ids, weights, (const bf16_t*)h, (const bf16_t*)w, bias, E, K, top, h_stride, sigmoid,
        scale);
  } else {
    route_plain_kernel<float><<<N, 256, E * 8, stream>>>(
        ids, weights, (const float*)h, (const float*)w, bias, E, K, top, h_stride, sigmoid,
        scale);
  }
}

void launch_moe_group(int* perm, int* offsets, int* tile_expert, int* tile_row, const int* ids,
                      int n, int E, hipStream_t stream) {
  auto kernel = tile_expert ? group_kernel<true> : group_kernel<false>;
  // a share has at least 1024 entries, a turn of its waves; one more workgroup for the lists
  const int shares = max(1, min(64, n / 1024));
  kernel<<<shares + 1, 1024, 18 * E * 4, stream>>>(perm, offsets, tile_expert, tile_row, ids, n, E);
}

// tt: 16 tokens at a time, or twice as many
void launch_experts_small(bool glu, const ExpertsArgs* a, int tt, hipStream_t stream) {
  const int per = glu ? 16 : 32;
  const dim3 grid((a->O + per - 1) / per, a->E);
  auto k = glu ? (tt == 1 ? experts_small_kernel<true, 2> : experts_small_kernel<true, 4>)
               : (tt == 1 ? experts_small_kernel<false, 2> : experts_small_kernel<false, 4>);
  k<<<grid, 256, 0, stream>>>(*a);
}

void launch_experts_f32(bool glu, const ExpertsArgs* a, hipStream_t stream) {
  const dim3 grid((a->entries + 3) / 4, (a->O + 63) / 64);
  auto k = glu ? experts_f32_kernel<true> : experts_f32_kernel<false>;
  k<<<grid, 256, 0, stream>>>(*a);
}

}  // extern "C"
