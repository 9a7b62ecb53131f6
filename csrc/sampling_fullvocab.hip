// Full-vocabulary token sampling (gfx950): temperature → optional grammar
// mask → exact top-k → top-p (nucleus) → inverse-CDF draw in token-id
// order; one workgroup per row, vocabularies up to 2^18 (Llama-3: 128256).
//
// The ≤512-entry LDS bitonic sampler (sampling.hip) covers the byte
// tokenizer; a real BPE vocabulary needs per-row selection over 128k
// entries.  Sorting is out at B≈1k rows; instead a threshold key (order-
// preserving uint32 of the logit) is found from histograms in LDS.  The first one
// is over m - x with 64 buckets an octave, so that neither the bulk of the logits nor
// their top meet in a few buckets; the bucket that holds the boundary is gathered into
// LDS and split by its keys until one key is left.  Buckets are weighted by 1 for
// top-k and by exp((x - m) / T) for top-p, and walked by a parallel scan.
//
// Every pass streams the row in 16-byte loads.  The draw sums 256 stripes of the row, each in
// token-id order, and walks the stripe with the target: the inverse CDF runs in token-id order
// and draws match the fp32 oracle (ops/reference.py softmax_sample) for a given uniform.  The
// weights of 64 tokens of every stripe are made at a time by all threads and added up by one
// thread a stripe, so that the order of the sums does not depend on the threads.
//
// Bound by the passes over the row: 20 us for the largest logit, 15 for the histogram of a top-k
// and 62 for that of a top-p (30 of it weights, 32 atomics), 16 to gather the bucket, 15 for the
// draw's sums, where 190 rows of 128256 in fp32 come from the memory-side cache.  Whole calls
// with other logits each time: 34 us greedy, 67 plain, 100 top-k, 153 top-p, 193 both; before 315,
// 428, 1135, 1305 and 1978 (thresholds by three histograms of key bits, whose few buckets met
// nearly all atomics, walked by one thread; draws by strides of a thread).  Floating masses
// instead of whole ones in the histogram took as long, a shared list of the bucket 25 us more.
//
// Semantics match the oracle:
//   greedy (T<=0): argmax, lowest index on ties
//   top-k:         keep {x >= kth-largest}   (ties at the k-th all kept)
//   top-p:         keep the minimal high-prob set whose exclusive
//                  cumulative <= p            (boundary-key ties all kept)
#include "common.h"

#define STRIPES 256
#define MOST_VOCAB (1 << 18)
#define OCTAVE 64       // first buckets: of m - x, per octave, from 2^-8 to 2^16
#define FIRST (24 * OCTAVE)
#define HEAD 12.f       // logits of at least exp(-HEAD) of the largest's weight come first
#define SPLIT 1024      // buckets of a further split
#define LIST 32         // keys of a bucket that a thread keeps in LDS

// order-preserving float -> uint32 key
__device__ __forceinline__ uint32_t f2key(float x) {
  uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key2f(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const bf16_t* p) { return bf2f(*p); }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Threads of a workgroup, and tokens of a stripe that are summed at a time.  With 1024 threads and
// 160 KB a CU has one row, and each step of a row ends in a wait for 16 waves: small vocabularies
// take 256 threads and 61 KB.  1024 and 256 threads, us: 512 rows of 600 greedy 10.7 and 5.7, plain
// 24.9 and 10.9, 16 rows of 4096 plain 14.2 and 9.8, top-p 29 and 24.  From there on only where
// the rows are more than the CUs: 512 rows of 8192 plain 30.8 and 15.6, but 16 rows top-p with a
// mask 32 and 39.
template <int THREADS, int TOKENS>
struct Form {
  static constexpr int WG = THREADS, WAVES = WG / 64, TILE = TOKENS;
  static constexpr int BUCKETS = (FIRST + WG - 1) / WG;  // of a thread
};

template <typename F>
struct Shared : F {
  uint32_t count[FIRST];
  unsigned long long mass[FIRST];  // in units of 2^-44: integer atomics are the fast ones
  union {
    uint32_t list[LIST][F::WG];
    float tile[2][STRIPES][F::TILE + 4];
  };
  float stripe[STRIPES], cdf[STRIPES + 1];
  double wave[F::WAVES];
  float red[F::WAVES];
  int red_i[F::WAVES];
  int n, pick;
  uint32_t lo, hi;
  double above;
};

#define UNIT 0x1p-44
// a weight, at most 1, in units; what is no number weighs nothing
__device__ __forceinline__ unsigned long long units(float w) {
  const float hi = floorf(w * 0x1p24f);  // exact, and so is the rest
  const float lo = (w - hi * 0x1p-24f) * 0x1p44f;
  return ((unsigned long long)(uint32_t)hi << 20) + (uint32_t)lo;
}

template <typename T, int WG>
struct Row {
  const T* x;
  const uint8_t* mask;  // or null
  int V;
  float m, invT;

  __device__ float weight(float v) const { return __expf((v - m) * invT); }

  // f(token, logit) for every allowed token, a thread's in rising order
  template <typename F>
  __device__ void each(F f) const {
    constexpr int N = 16 / sizeof(T), AHEAD = 4;
    auto one = [&](int i, float v) {
      if (!mask || mask[i]) f(i, v);
    };
    auto all = [&](int i, u32x4 v) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        const uint32_t bits = N == 4 ? v[e & 3] : (e & 1) ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16;
        one(i + e, __uint_as_float(bits));
      }
    };
    int i = 0;
    if ((uintptr_t)x % 16 == 0) {
      const int whole = V / (WG * N) * WG * N;
      for (; i + AHEAD * WG * N <= whole; i += AHEAD * WG * N) {
        u32x4 v[AHEAD];
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
          v[a] = *(const u32x4*)(x + i + (a * WG + threadIdx.x) * N);
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) all(i + (a * WG + threadIdx.x) * N, v[a]);
      }
      for (; i < whole; i += WG * N)
        all(i + threadIdx.x * N, *(const u32x4*)(x + i + threadIdx.x * N));
    }
    for (i += threadIdx.x; i < V; i += WG) one(i, ldf(x + i));
  }

  // bucket of a logit: 0 holds the largest
  __device__ int bucket(float v) const {
    const int b = (int)(__float_as_uint(m - v) >> 17) - ((127 - 8) << 6);
    return min(max(b, 0), FIRST - 1);
  }
};
static_assert(OCTAVE == 64, "bucket() takes 6 bits of the mantissa");

// The first of ``n`` (at most FIRST) buckets whose sum with those before and ``above`` reaches
// target, and the sum before it; -1: none does.
template <bool BY_MASS, typename S>
__device__ int find_bucket(S& s, int n, double target, double* above) {
  constexpr int PER = S::BUCKETS;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double w[PER], sum = 0.0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = PER * threadIdx.x + j;
    w[j] = i >= n ? 0.0 : BY_MASS ? s.mass[i] * UNIT : (double)s.count[i];
    sum += w[j];
  }
  double upto = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double v = __shfl_up(upto, off, 64);
    if (lane >= off) upto += v;
  }
  if (lane == 63) s.wave[wid] = upto;
  if (threadIdx.x == 0) s.n = 1 << 30;
  __syncthreads();
  double before = *above;
  for (int i = 0; i < wid; ++i) before += s.wave[i];
  before += upto - sum;
  int mine = n;
  double mine_before = 0.0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const double after = before + w[j];
    if (mine == n && after >= target) {
      mine = min(n, (int)(PER * threadIdx.x) + j);
      mine_before = before;
    }
    before = after;
  }
  if (mine < n) atomicMin(&s.n, mine);
  __syncthreads();
  const int got = s.n;
  if (mine == got) s.above = mine_before;
  __syncthreads();
  if (got < n) *above = s.above;
  return got < n ? got : -1;
}

// Splits the keys [lo, hi] among those that each_key(f) hands out until one is left: the one at
// which the sum from the top reaches target.
template <bool BY_MASS, typename S, typename R, typename E>
__device__ uint32_t split_keys(S& s, const R& row, uint32_t lo, uint32_t hi,
                               double above, double target, E each_key) {
  for (;;) {
    const uint32_t range = hi - lo;
    const int shift = range < SPLIT ? 0 : 32 - __builtin_clz(range) - 10;
    const int n = (int)(range >> shift) + 1;
    for (int i = threadIdx.x; i < n; i += S::WG) {
      s.count[i] = 0;
      s.mass[i] = 0;
    }
    __syncthreads();
    each_key([&](uint32_t key) {
      if (key < lo || key > hi) return;
      const uint32_t b = (hi - key) >> shift;
      if (BY_MASS)
        atomicAdd(&s.mass[b], units(row.weight(key2f(key))));
      else
        atomicAdd(&s.count[b], 1u);
    });
    __syncthreads();
    int b = find_bucket<BY_MASS>(s, n, target, &above);
    if (b < 0) b = n - 1;
    hi -= (uint32_t)b << shift;
    const uint32_t width = (1u << shift) - 1;
    if (hi - lo > width) lo = hi - width;
    if (shift == 0) return hi;
  }
}

template <typename S>
__device__ double block_total(S& s, double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) s.wave[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < S::WAVES; ++w) t += s.wave[w];
  __syncthreads();
  return t;
}

// Histograms over m - x up to ``far``; the mass of the others: a boundary is seldom among
// them, and their atomics take most of the time.
template <bool BY_MASS, typename S, typename R>
__device__ float fill(S& s, const R& row, float far) {
  for (int i = threadIdx.x; i < FIRST; i += S::WG) {
    s.count[i] = 0;
    s.mass[i] = 0;
  }
  __syncthreads();
  float rest = 0.f;
  row.each([&](int, float v) {
    const float w = BY_MASS ? row.weight(v) : 0.f;
    if (row.m - v > far) {
      rest += w;
      return;
    }
    const int b = row.bucket(v);
    if (BY_MASS)
      atomicAdd(&s.mass[b], units(w));
    else
      atomicAdd(&s.count[b], 1u);
  });
  __syncthreads();
  return rest;
}

// The key at which the sum from the largest logit down reaches target, which is ``part`` of all
// weights if it is given; 0: nowhere.  ``plain``: all logits are numbers.
template <bool BY_MASS, typename S, typename R>
__device__ uint32_t boundary(S& s, const R& row, double target, double part, bool plain) {
  if (target <= 0.0) return f2key(row.m);  // reached before the first, which is kept all the same
  auto stream = [&](auto f) { row.each([&](int, float v) { f(f2key(v)); }); };
  if (!plain) return split_keys<BY_MASS>(s, row, 0u, 0xffffffffu, 0.0, target, stream);
  double above = 0.0;
  const float rest = fill<BY_MASS>(s, row, HEAD / row.invT);
  if (part > 0.0) {
    double all = 0.0;
    for (int i = threadIdx.x; i < FIRST; i += S::WG) all += s.mass[i] * UNIT;
    target = part * block_total(s, all + rest);
    if (target <= 0.0) return f2key(row.m);
  }
  int b = find_bucket<BY_MASS>(s, FIRST, target, &above);
  if (b < 0) {  // beyond the head
    fill<BY_MASS>(s, row, INFINITY);
    above = 0.0;
    b = find_bucket<BY_MASS>(s, FIRST, target, &above);
    if (b < 0) return 0;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    s.n = 0;
    s.lo = 0xffffffffu;
    s.hi = 0;
  }
  __syncthreads();
  uint32_t lo = 0xffffffffu, hi = 0;
  int n = 0;  // this thread's, in a column of the list
  row.each([&](int, float v) {
    if (row.bucket(v) != b) return;
    const uint32_t key = f2key(v);
    lo = min(lo, key);
    hi = max(hi, key);
    if (n < LIST) s.list[n][threadIdx.x] = key;
    ++n;
  });
  if (n) {
    atomicMin(&s.lo, lo);
    atomicMax(&s.hi, hi);
    if (n > LIST) s.n = 1;
  }
  __syncthreads();
  lo = s.lo;
  hi = s.hi;
  const bool fits = s.n == 0;
  __syncthreads();
  if (!fits) return split_keys<BY_MASS>(s, row, lo, hi, above, target, stream);
  return split_keys<BY_MASS>(s, row, lo, hi, above, target, [&](auto f) {
    for (int i = 0; i < n; ++i) f(s.list[i][threadIdx.x]);
  });
}

template <typename T, typename F>
__global__ __launch_bounds__(F::WG) void sample_fullvocab_kernel(
    int64_t* __restrict__ out,           // [B]
    const T* __restrict__ logits,        // [B, V]
    const float* __restrict__ temps,     // [B]
    const int64_t* __restrict__ top_ks,  // [B] (0 = off)
    const float* __restrict__ top_ps,    // [B]
    const float* __restrict__ uniforms,  // [B] in [0,1)
    const uint8_t* __restrict__ mask,    // [M, V] bool, may be null
    const int32_t* __restrict__ mask_map,// [B] row -> mask row (-1 = none)
    const int V) {
  constexpr int WG = F::WG, WAVES = F::WAVES, TILE = F::TILE;
  __shared__ Shared<F> s;
  const int n_row = blockIdx.x, t = threadIdx.x, lane = t & 63, wid = t >> 6;
  // compact masks: only constrained rows carry one (a dense [B,V] mask at
  // B=1k, V=128k would be 128 MB of pinned staging per step)
  const bool masked = mask && mask_map && mask_map[n_row] >= 0;
  const float Tmp = temps[n_row];
  const bool greedy = Tmp <= 0.f;
  Row<T, WG> row = {logits + (int64_t)n_row * V,
                masked ? mask + (int64_t)mask_map[n_row] * V : nullptr, V, 0.f,
                greedy ? 1.f : 1.f / Tmp};

  // ---- the largest allowed logit, the lowest token that has it, and whether all are numbers
  float mx = -3.4e38f;
  int best = V, odd = 0;
  row.each([&](int i, float v) {
    if (v > mx) {
      mx = v;
      best = i;
    } else if (v == mx) {
      best = min(best, i);
    }
    odd |= !(v < INFINITY);
  });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float v = __shfl_xor(mx, off, 64);
    const int i = __shfl_xor(best, off, 64);
    if (v > mx || (v == mx && i < best)) best = i;
    mx = fmaxf(mx, v);
  }
  const bool odd_wave = __any(odd);
  if (lane == 0) {
    s.red[wid] = mx;
    s.red_i[wid] = best;
    s.cdf[wid] = odd_wave;
  }
  __syncthreads();
  bool plain = true;
  for (int w = 0; w < WAVES; ++w) {
    if (s.red[w] > mx || (s.red[w] == mx && s.red_i[w] < best)) best = s.red_i[w];
    mx = fmaxf(mx, s.red[w]);
    plain &= s.cdf[w] == 0.f;
  }
  __syncthreads();
  row.m = mx;
  if (greedy) {
    if (t == 0) out[n_row] = best < V ? best : 0;
    return;
  }

  // ---- top-k, then top-p: kept = {key >= kmin}
  uint32_t kmin = 0;
  const int64_t tk = top_ks[n_row];
  const float p = top_ps[n_row];
  const bool by_k = tk > 0 && tk < V, by_p = p < 1.f;
  if (by_k) kmin = boundary<false>(s, row, (double)tk, 0.0, plain);
  if (by_p) {
    double target = p;
    if (by_k || !plain) {  // of what is kept so far
      float kept = 0.f;
      row.each([&](int, float v) {
        if (f2key(v) >= kmin) kept += row.weight(v);
      });
      target = (double)p * (float)block_total(s, kept);
    }
    // all keys above the boundary are kept: the histograms need not know kmin
    const uint32_t pmin =
        boundary<true>(s, row, target, by_k || !plain ? 0.0 : (double)p, plain);
    if (pmin > kmin) kmin = pmin;
  }

  // ---- inverse-CDF draw in token-id order over the kept set.
  // Stripe n is tokens [n * stride, (n + 1) * stride).
  const int stride = (V + STRIPES - 1) / STRIPES;
  constexpr int PER = STRIPES * TILE / WG, ROWS = WG / TILE;  // a thread's tokens of a tile
  // token of the thread's k-th of a tile: k * ROWS stripes on
  const int r = t / TILE, c = t % TILE, i_first = r * stride + c;
  float ahead[PER];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int k = 0; k < PER; ++k)
      ahead[k] = ldf(row.x + min(k * ROWS * stride + j0 + i_first, V - 1));
  };
  // comparing logits is comparing keys, but for zeros and what is no number
  const float least = key2f(kmin);
  const bool by_value = kmin == 0 || (least == least && least != 0.f);
  const float from = kmin == 0 ? -INFINITY : least;
  const bool even = V == STRIPES * stride;  // no stripe is shorter
  float mine = 0.f;
  fetch(0);
  for (int j0 = 0; j0 < stride; j0 += TILE) {
    float(*tile)[TILE + 4] = s.tile[j0 / TILE % 2];
    if (even && by_value && plain && !row.mask && j0 + TILE <= stride) {
#pragma unroll
      for (int k = 0; k < PER; ++k)
        tile[k * ROWS + r][c] = ahead[k] >= from ? row.weight(ahead[k]) : 0.f;
    } else {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int i = k * ROWS * stride + j0 + i_first;
        const bool in = j0 + c < stride && i < V && f2key(ahead[k]) >= kmin &&
                        !(row.mask && !row.mask[i]);
        tile[k * ROWS + r][c] = in ? row.weight(ahead[k]) : 0.f;
      }
    }
    if (j0 + TILE < stride) fetch(j0 + TILE);
    __syncthreads();  // the other tile is added up before it is written again
    if (t < STRIPES) {
      float4 w[TILE / 4];
#pragma unroll
      for (int j = 0; j < TILE / 4; ++j) w[j] = *(const float4*)&tile[t][4 * j];
#pragma unroll
      for (int j = 0; j < TILE / 4; ++j) mine = mine + w[j].x + w[j].y + w[j].z + w[j].w;
    }
  }
  if (t < STRIPES) s.stripe[t] = mine;
  if (t == 0) s.pick = s.n = -1;
  __syncthreads();
  constexpr int STEP = 32;  // one thread's LDS reads in flight
  if (t == 0) {
    float sum = 0.f;
    s.cdf[0] = 0.f;
    for (int i = 0; i < STRIPES; i += STEP) {
      float w[STEP];
#pragma unroll
      for (int e = 0; e < STEP; ++e) w[e] = s.stripe[i + e];
#pragma unroll
      for (int e = 0; e < STEP; ++e) s.cdf[i + e + 1] = sum += w[e];
    }
  }
  __syncthreads();
  const float target = uniforms[n_row] * s.cdf[STRIPES];
  // exactly one stripe satisfies prefix <= target < prefix + mine
  // (mine > 0 guaranteed for the owner since the CDF strictly increases
  // across it); fp edge cases fall through to the fallback below
  if (t < STRIPES && mine > 0.f && s.cdf[t] <= target && target < s.cdf[t + 1]) s.n = t;
  __syncthreads();
  const int n = s.n;
  __syncthreads();
  if (n >= 0) {
    // the stripe's weights, added up in order by one thread until they exceed the target;
    // its last kept token if rounding lets none do so
    float* const buf = &s.tile[0][0][0];
    static_assert(sizeof(s.tile) >= 4 * (MOST_VOCAB / STRIPES + STEP), "a stripe fits");
    const int i0 = n * stride, here = min(stride, V - i0);
    int last = -1;
    for (int j = t; j < (here + STEP - 1) / STEP * STEP; j += WG) {
      float w = 0.f;
      if (j < here && !(row.mask && !row.mask[i0 + j])) {
        const float v = ldf(row.x + i0 + j);
        if (f2key(v) >= kmin) {
          w = row.weight(v);
          last = i0 + j;
        }
      }
      buf[j] = w;
    }
    if (last >= 0) atomicMax(&s.pick, last);
    __syncthreads();
    if (t == 0) {
      float cum = s.cdf[n];
      int first = STEP;
      for (int j = 0; j < here && first == STEP; j += STEP) {
        float w[STEP];
#pragma unroll
        for (int e = 0; e < STEP; e += 4) *(float4*)(w + e) = *(const float4*)(buf + j + e);
#pragma unroll
        for (int e = 0; e < STEP; ++e) {
          cum += w[e];
          if (first == STEP && cum > target) first = e;
        }
        if (first < STEP) s.pick = i0 + j + first;
      }
    }
  }
  __syncthreads();
  if (t == 0 && s.pick < 0) {
    // fallback (target == total to fp precision, or an empty kept set):
    // the last kept token, matching searchsorted's clamp in the oracle; else the last allowed one
    int last = -1;
    for (int i = V - 1; i >= 0; --i) {
      if (row.mask && !row.mask[i]) continue;
      if (last < 0) last = i;
      if (f2key(ldf(row.x + i)) < kmin) continue;
      last = i;
      break;
    }
    s.pick = max(last, 0);
  }
  __syncthreads();
  if (t == 0) out[n_row] = s.pick;
}

template <typename T>
static void launch(int64_t* out, const T* logits, const float* temps, const int64_t* top_ks,
                   const float* top_ps, const float* uniforms, const uint8_t* mask,
                   const int32_t* mask_map, int B, int V, hipStream_t stream) {
  using Small = Form<256, 16>;
  using Large = Form<1024, 64>;
  const bool small = V <= 4096 || (V <= 8192 && B > 256);
  auto kernel = small ? sample_fullvocab_kernel<T, Small> : sample_fullvocab_kernel<T, Large>;
  kernel<<<B, small ? Small::WG : Large::WG, 0, stream>>>(out, logits, temps, top_ks, top_ps,
                                                          uniforms, mask, mask_map, V);
}

extern "C" void launch_sample_fullvocab(int64_t* out, const void* logits, bool bf16,
                             const float* temps, const int64_t* top_ks,
                             const float* top_ps, const float* uniforms,
                             const uint8_t* mask, const int32_t* mask_map,
                             int B, int V, hipStream_t stream) {
  if (bf16)
    launch(out, (const bf16_t*)logits, temps, top_ks, top_ps, uniforms, mask, mask_map, B, V, stream);
  else
    launch(out, (const float*)logits, temps, top_ks, top_ps, uniforms, mask, mask_map, B, V, stream);
}
