// Full-vocabulary token sampling (gfx950): temperature → optional grammar
// mask → exact top-k → top-p (nucleus) → inverse-CDF draw in token-id
// order; one workgroup per row, or several for few rows of large vocabularies ("rows in chunks"), up to
// 2^18 tokens (Llama-3: 128256).
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
// A workgroup a row is bound by its passes over the row.  190 rows of 128256 in fp32, other logits each
// time, whole calls: 25 us greedy, 48 plain, 79 top-k, 95 top-p, 135 both (26, 58, 97, 168 and 238 with
// calls of functions, which take a row and LDS by reference: their loads and atomics then go by
// unknown memory and wait for both kinds); before 315,
// 428, 1135, 1305 and 1978 (thresholds by three histograms of key bits, whose few buckets met
// nearly all atomics, walked by one thread; draws by strides of a thread).  Floating masses
// instead of whole ones in the histogram took as long, a shared list of the bucket 25 us more.
//
// Semantics match the oracle:
//   greedy (T<=0): argmax, lowest index on ties
//   top-k:         keep {x >= kth-largest}   (ties at the k-th all kept)
//   top-p:         keep the minimal high-prob set whose exclusive
//                  cumulative <= p            (boundary-key ties all kept)
#include <type_traits>

#include "common.h"

#define STRIPES 256
#define MOST_VOCAB (1 << 18)
#define OCTAVE 64       // first buckets: of m - x, per octave, from 2^-8 to 2^16
#define FIRST (24 * OCTAVE)
#define HEAD 12.f       // logits of at least exp(-HEAD) of the largest's weight come first
#define SPLIT 1024      // buckets of a further split
#define LIST 32         // keys of a bucket that a thread keeps in LDS
#define KEYS 2048       // of the list of a row in chunks
#define RANKED 320      // of them at most are compared with one another

// order-preserving float -> uint32 key
__device__ __forceinline__ uint32_t f2key(float x) {
  uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key2f(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

#define INLINE __device__ __forceinline__
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
    float buffer[2 * STRIPES * (F::TILE + 4)];  // of the drawn stripe
    struct {
      alignas(16) uint32_t key[KEYS];  // of a row in chunks
      unsigned long long key_mass[KEYS];
    };
  };
  float stripe[STRIPES], cdf[STRIPES + 1];
  double wave[F::WAVES];
  float red[F::WAVES];
  int red_i[F::WAVES], red_odd[F::WAVES];
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
  INLINE void each(F f) const {
    each(0, V, f);
  }
  // likewise of tokens i0 .. i1 - 1
  template <typename F>
  INLINE void each(int i0, int i1, F f) const {
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
    int i = i0;
    if ((uintptr_t)(x + i0) % 16 == 0) {
      const int whole = i0 + (i1 - i0) / N * N;
      for (; i + AHEAD * WG * N <= whole; i += AHEAD * WG * N) {
        u32x4 v[AHEAD];
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
          v[a] = *(const u32x4*)(x + i + (a * WG + threadIdx.x) * N);
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) all(i + (a * WG + threadIdx.x) * N, v[a]);
      }
      if (i < whole) {  // a last turn of fewer
        u32x4 v[AHEAD];
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
          v[a] = *(const u32x4*)(x + min(i + (int)(a * WG + threadIdx.x) * N, whole - N));
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
          const int at = i + (a * WG + threadIdx.x) * N;
          if (at < whole) all(at, v[a]);
        }
      }
      i = whole;
    }
    for (i += threadIdx.x; i < i1; i += WG) one(i, ldf(x + i));
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
INLINE int find_bucket(S& s, int n, double target, double* above) {
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
INLINE uint32_t split_keys(S& s, const R& row, uint32_t lo, uint32_t hi,
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
INLINE double block_total(S& s, double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) s.wave[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < S::WAVES; ++w) t += s.wave[w];
  __syncthreads();
  return t;
}

// The largest of the threads' logits, the lowest token among equals, whether one is odd
template <typename S>
INLINE void block_max(S& s, float& mx, int& best, int& odd) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float v = __shfl_xor(mx, off, 64);
    const int i = __shfl_xor(best, off, 64);
    if (v > mx || (v == mx && i < best)) best = i;
    mx = fmaxf(mx, v);
  }
  const int wid = threadIdx.x >> 6;
  const bool odd_wave = __any(odd);
  if ((threadIdx.x & 63) == 0) {
    s.red[wid] = mx;
    s.red_i[wid] = best;
    s.red_odd[wid] = odd_wave;
  }
  __syncthreads();
  odd = 0;
  for (int w = 0; w < S::WAVES; ++w) {
    if (s.red[w] > mx || (s.red[w] == mx && s.red_i[w] < best)) best = s.red_i[w];
    mx = fmaxf(mx, s.red[w]);
    odd |= s.red_odd[w];
  }
  __syncthreads();
}

// Histograms over m - x up to ``far``; the mass of the others: a boundary is seldom among
// them, and their atomics take most of the time.
template <bool BY_MASS, typename S, typename R>
INLINE float fill(S& s, const R& row, float far) {
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
INLINE uint32_t boundary(S& s, const R& row, double target, double part, bool plain) {
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

struct SampleArgs {
  int64_t* out;            // [B]
  const void* logits;      // [B, V]
  const float* temps;      // [B]
  const int64_t* top_ks;   // [B] (0 = off)
  const float* top_ps;     // [B]
  const float* uniforms;   // [B] in [0,1)
  const uint8_t* mask;     // [M, V] bool, may be null
  const int32_t* mask_map; // [B] row -> mask row (-1 = none)
  int B, V;
};

// compact masks: only constrained rows carry one (a dense [B,V] mask at
// B=1k, V=128k would be 128 MB of pinned staging per step)
template <typename T, int WG>
INLINE Row<T, WG> row_of(const SampleArgs& a, int n) {
  const bool masked = a.mask && a.mask_map && a.mask_map[n] >= 0;
  const float temp = a.temps[n];
  return {(const T*)a.logits + (int64_t)n * a.V,
          masked ? a.mask + (int64_t)a.mask_map[n] * a.V : nullptr, a.V, 0.f,
          temp <= 0.f ? 1.f : 1.f / temp};
}

// ---- inverse-CDF draw in token-id order from the stripes' sums, ``mine`` of the t-th thread's
template <typename S, typename R>
INLINE void draw(S& s, const SampleArgs& a, const R& row, int n_row, uint32_t kmin,
                     float mine) {
  constexpr int WG = S::WG;
  const int t = threadIdx.x, V = row.V, stride = (V + STRIPES - 1) / STRIPES;
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
  const float target = a.uniforms[n_row] * s.cdf[STRIPES];
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
    float* const buf = s.buffer;
    static_assert(sizeof(s.buffer) >= 4 * (MOST_VOCAB / STRIPES + STEP), "a stripe fits");
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
        float w[STEP], upto = cum;
#pragma unroll
        for (int e = 0; e < STEP; e += 4) *(float4*)(w + e) = *(const float4*)(buf + j + e);
#pragma unroll
        for (int e = 0; e < STEP; ++e) upto += w[e];
        if (!(upto <= target))  // the same sums again: weights are not negative
          for (int e = 0; e < STEP && first == STEP; ++e)
            if ((cum += buf[j + e]) > target) first = e;
        cum = upto;
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
  if (t == 0) a.out[n_row] = s.pick;
}

// ---- rows in chunks
//
// Few rows of large vocabularies: a row's 256 stripes go to ``chunks`` workgroups in launches of their
// own, so that they have the whole chip.
//   1 the largest logit of a chunk
//   2 a chunk's histograms, added to the row's
//   3 the boundary's bucket from those, by every workgroup; its keys into the row's list
//   4 a workgroup a row: the least key that is kept, from the list
//   5 the sums of a chunk's stripes
//   6 a workgroup a row: the draw
// All that workgroups share are whole numbers or added up in a fixed order, so that they agree.  A
// row that this does not fit (logits that are no numbers, a boundary beyond the head or among more
// keys than the list has) is taken as a whole in launch 4.
// 16 x 128256 of plain, top-k, top-p and greedy rows in turns 63 us, by a workgroup a row 84.
#define SPLIT_VOCAB 100000
#define LEAST_CHUNKS 16
#define MOST_CHUNKS 32

enum Mode { NO_LIST, BY_LIST, WHOLE };

struct RowPlan {
  int mode;        // where the least kept key comes from: kmin, the list, the whole row
  int n;           // keys that the list was asked to take
  uint32_t kmin;
  double above, target;  // of the list's keys: top-k's, or top-p's without a top-k
  float m;
  int best, plain;
};

__device__ __forceinline__ bool left_whole(const RowPlan& plan) {
  return plan.mode == WHOLE || (plan.mode == BY_LIST && plan.n > KEYS);
}

// A row's state between the launches
struct RowState {
  RowPlan plan;
  double rest[MOST_CHUNKS];
  float chunk_max[MOST_CHUNKS];
  int chunk_best[MOST_CHUNKS], chunk_odd[MOST_CHUNKS];
  float stripe[STRIPES];
  uint32_t list[KEYS];
  uint32_t count[FIRST];
  unsigned long long mass[FIRST];
};

typedef Form<256, 64> ChunkForm;

struct ChunkShared : ChunkForm {
  union {
    struct {
      uint32_t count[FIRST];
      unsigned long long mass[FIRST];
    };
    float tile[2][STRIPES / LEAST_CHUNKS][TILE + 4];
  };
  uint32_t keys[KEYS];
  double wave[WAVES];
  float red[WAVES];
  int red_i[WAVES], red_odd[WAVES];
  int n, base;
  uint32_t lo, hi;
  double above;
};

struct Chunk {
  int row, at, stride, stripes, i0, i1;
};
__device__ __forceinline__ Chunk chunk_of(const SampleArgs& a, int chunks) {
  Chunk c;
  c.row = blockIdx.x / chunks;
  c.at = blockIdx.x - c.row * chunks;
  c.stride = (a.V + STRIPES - 1) / STRIPES;
  c.stripes = STRIPES / chunks;
  c.i0 = min(a.V, c.at * c.stripes * c.stride);
  c.i1 = min(a.V, c.i0 + c.stripes * c.stride);
  return c;
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_max_kernel(const SampleArgs a, RowState* states,
                                                        const int chunks) {
  __shared__ ChunkShared s;
  const Chunk c = chunk_of(a, chunks);
  const Row<T, 256> row = row_of<T, 256>(a, c.row);
  RowState& state = states[c.row];
  for (int i = c.at * 256 + threadIdx.x; i < FIRST; i += chunks * 256) {
    state.count[i] = 0;
    state.mass[i] = 0;
  }
  if (c.at == 0 && threadIdx.x == 0) state.plan.n = 0;
  float mx = -3.4e38f;
  int best = a.V, odd = 0;
  row.each(c.i0, c.i1, [&](int i, float v) {
    if (v > mx) {
      mx = v;
      best = i;
    } else if (v == mx) {
      best = min(best, i);
    }
    odd |= !(v < INFINITY);
  });
  block_max(s, mx, best, odd);
  if (threadIdx.x == 0) {
    state.chunk_max[c.at] = mx;
    state.chunk_best[c.at] = best;
    state.chunk_odd[c.at] = odd;
  }
}

// the row's largest logit, the lowest token that has it, and whether all are numbers
template <typename R>
INLINE bool whole_max(const RowState& state, int chunks, R& row, int* best) {
  float mx = -3.4e38f;
  int at = row.V, odd = 0;
  for (int i = 0; i < chunks; ++i) {
    const float v = state.chunk_max[i];
    const int b = state.chunk_best[i];
    if (v > mx || (v == mx && b < at)) at = b;
    mx = fmaxf(mx, v);
    odd |= state.chunk_odd[i];
  }
  row.m = mx;
  *best = at;
  return !odd;
}

struct Wants {
  bool greedy, by_k, by_p;
  double k;
  float p;
};
__device__ __forceinline__ Wants wants_of(const SampleArgs& a, int n) {
  Wants w;
  const int64_t tk = a.top_ks[n];
  w.greedy = a.temps[n] <= 0.f;
  w.p = a.top_ps[n];
  w.by_k = tk > 0 && tk < a.V;
  w.by_p = w.p < 1.f;
  w.k = (double)tk;
  return w;
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_histogram_kernel(const SampleArgs a,
                                                              RowState* states, const int chunks) {
  __shared__ ChunkShared s;
  const Chunk c = chunk_of(a, chunks);
  const Wants want = wants_of(a, c.row);
  if (want.greedy || !(want.by_k || want.by_p)) return;
  Row<T, 256> row = row_of<T, 256>(a, c.row);
  RowState& state = states[c.row];
  int best;
  if (!whole_max(state, chunks, row, &best)) return;
  for (int i = threadIdx.x; i < FIRST; i += 256) {
    s.count[i] = 0;
    s.mass[i] = 0;
  }
  __syncthreads();
  const float far = HEAD / row.invT;
  float rest = 0.f;
  row.each(c.i0, c.i1, [&](int, float v) {
    const float w = want.by_p ? row.weight(v) : 0.f;
    if (row.m - v > far) {
      rest += w;
      return;
    }
    const int b = row.bucket(v);
    if (want.by_p) atomicAdd(&s.mass[b], units(w));
    if (want.by_k) atomicAdd(&s.count[b], 1u);
  });
  const double all = block_total(s, (double)rest);
  if (threadIdx.x == 0) state.rest[c.at] = all;
  __syncthreads();
  for (int i = threadIdx.x; i < FIRST; i += 256) {
    if (s.count[i]) atomicAdd(&state.count[i], s.count[i]);
    if (s.mass[i]) atomicAdd(&state.mass[i], s.mass[i]);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_keys_kernel(const SampleArgs a, RowState* states,
                                                         const int chunks) {
  __shared__ ChunkShared s;
  const Chunk c = chunk_of(a, chunks);
  const Wants want = wants_of(a, c.row);
  Row<T, 256> row = row_of<T, 256>(a, c.row);
  RowState& state = states[c.row];
  RowPlan plan = {NO_LIST, 0, 0, 0.0, 0.0, 0.f, 0, 0};
  plan.plain = whole_max(state, chunks, row, &plan.best);
  plan.m = row.m;
  int first = 0, last = -1;  // buckets
  if (!want.greedy && (want.by_k || want.by_p)) {
    if (plan.plain) {
      for (int i = threadIdx.x; i < FIRST; i += 256) {
        s.count[i] = state.count[i];
        s.mass[i] = state.mass[i];
      }
      __syncthreads();
      plan.mode = BY_LIST;
      plan.target = want.k;
      if (want.by_k) {
        last = find_bucket<false>(s, FIRST, want.k, &plan.above);
        if (last >= 0 && !want.by_p) first = last;
        // with both, the nucleus is among the keys from the largest down
        if (last >= 0 && s.count[last] + (want.by_p ? plan.above : 0.0) > KEYS) last = -1;
        if (want.by_p) plan.above = 0.0;
      } else {
        double all = 0.0;
        for (int i = threadIdx.x; i < FIRST; i += 256) all += s.mass[i] * UNIT;
        if (threadIdx.x < chunks) all += state.rest[threadIdx.x];
        plan.target = (double)want.p * block_total(s, all);
        if (plan.target <= 0.0) {  // reached before the first, which is kept all the same
          plan.mode = NO_LIST;
          plan.kmin = f2key(row.m);
        } else {
          first = last = find_bucket<true>(s, FIRST, plan.target, &plan.above);
        }
      }
      if (plan.mode == BY_LIST && last < 0) plan.mode = WHOLE;
    } else {
      plan.mode = WHOLE;
    }
  }
  if (c.at == 0 && threadIdx.x == 0) {
    const RowPlan& p = plan;
    RowPlan& to = state.plan;  // all but n, which others count up
    to.mode = p.mode; to.kmin = p.kmin; to.above = p.above; to.target = p.target;
    to.m = p.m; to.best = p.best; to.plain = p.plain;
  }
  if (plan.mode != BY_LIST) return;
  if (threadIdx.x == 0) s.n = 0;
  __syncthreads();
  row.each(c.i0, c.i1, [&](int, float v) {
    const int b = row.bucket(v);
    if (b < first || b > last) return;
    const int at = atomicAdd(&s.n, 1);
    if (at < KEYS) s.keys[at] = f2key(v);
  });
  __syncthreads();
  const int n = s.n;
  if (n == 0) return;
  if (threadIdx.x == 0) s.base = atomicAdd(&state.plan.n, n);
  __syncthreads();
  for (int i = threadIdx.x; i < n && s.base + i < KEYS; i += 256) state.list[s.base + i] = s.keys[i];
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_sums_kernel(const SampleArgs a, RowState* states,
                                                         const int chunks) {
  constexpr int TILE = ChunkForm::TILE;
  __shared__ ChunkShared s;
  const Chunk c = chunk_of(a, chunks);
  const Wants want = wants_of(a, c.row);
  if (want.greedy) return;
  Row<T, 256> row = row_of<T, 256>(a, c.row);
  RowState& state = states[c.row];
  const RowPlan plan = state.plan;
  const int t = threadIdx.x;
  row.m = plan.m;
  if (left_whole(plan)) return;
  const uint32_t kmin = plan.kmin;
  // stripes' weights by all threads, 64 tokens of each at a time, added up by a thread a stripe
  const int r = t / TILE, col = t % TILE;
  constexpr int ROWS = 256 / TILE, MOST = STRIPES / LEAST_CHUNKS / ROWS;
  const float least = key2f(kmin);
  const bool by_value = kmin == 0 || (least == least && least != 0.f);
  const float from = kmin == 0 ? -INFINITY : least;
  float ahead[MOST], mine = 0.f;
  auto fetch = [&](int j0) {
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (k * ROWS < c.stripes)
        ahead[k] = ldf(row.x + min(c.i0 + (k * ROWS + r) * c.stride + j0 + col, a.V - 1));
  };
  fetch(0);
  for (int j0 = 0; j0 < c.stride; j0 += TILE) {
    float(*tile)[TILE + 4] = s.tile[j0 / TILE % 2];
#pragma unroll
    for (int k = 0; k < MOST; ++k) {
      if (k * ROWS >= c.stripes) break;
      const int i = c.i0 + (k * ROWS + r) * c.stride + j0 + col;
      // comparing logits is comparing keys, but for zeros and what is no number
      const bool keep = by_value && plan.plain ? ahead[k] >= from : f2key(ahead[k]) >= kmin;
      const bool in = j0 + col < c.stride && i < a.V && keep && !(row.mask && !row.mask[i]);
      tile[k * ROWS + r][col] = in ? row.weight(ahead[k]) : 0.f;
    }
    if (j0 + TILE < c.stride) fetch(j0 + TILE);
    __syncthreads();  // the other tile is added up before it is written again
    if (t < c.stripes) {
      float4 w[TILE / 4];
#pragma unroll
      for (int j = 0; j < TILE / 4; ++j) w[j] = *(const float4*)&tile[t][4 * j];
#pragma unroll
      for (int j = 0; j < TILE / 4; ++j) mine = mine + w[j].x + w[j].y + w[j].z + w[j].w;
    }
  }
  if (t < c.stripes) state.stripe[c.at * c.stripes + t] = mine;
}

struct DrawShared : ChunkForm {
  alignas(16) float buffer[MOST_VOCAB / STRIPES + 64];
  float stripe[STRIPES], cdf[STRIPES + 1];
  int n, pick;
};

template <typename T>
__global__ __launch_bounds__(256) void draw_kernel(const SampleArgs a, const RowState* states) {
  __shared__ DrawShared s;
  const int n_row = blockIdx.x;
  const RowState& state = states[n_row];
  const RowPlan plan = state.plan;
  if (a.temps[n_row] <= 0.f) {
    if (threadIdx.x == 0) a.out[n_row] = plan.best < a.V ? plan.best : 0;
    return;
  }
  if (left_whole(plan)) return;
  Row<T, 256> row = row_of<T, 256>(a, n_row);
  row.m = plan.m;
  draw(s, a, row, n_row, plan.kmin, state.stripe[threadIdx.x]);
}

// The key of a list at which the sum from the top, with what is ``above``, reaches target, the
// least one if rounding lets none do so.  A thread compares its key with all others, which takes
// 33 ns a key; the two rounds of split_keys take about 12 us whatever the list: RANKED keys.
template <bool BY_MASS, typename S>
INLINE uint32_t rank_keys(S& s, int n, double above, double target) {
  if (threadIdx.x == 0) s.lo = 0xffffffffu;
  __syncthreads();
  uint32_t least = 0xffffffffu, at = 0;
  bool found = false;
  for (int i = threadIdx.x; i < n; i += S::WG) {
    const uint32_t key = s.key[i];
    unsigned long long higher = 0, same = 0;
    for (int j = 0; j < n; j += 4) {
      const u32x4 k = *(const u32x4*)&s.key[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // the units behind the last key are 0
        const unsigned long long w = BY_MASS ? s.key_mass[j + e] : j + e < n;
        higher += k[e] > key ? w : 0;
        same += k[e] == key ? w : 0;
      }
    }
    const double unit = BY_MASS ? UNIT : 1.0;
    const double before = above + (double)higher * unit;
    if (before < target && before + (double)same * unit >= target) {
      found = true;
      at = key;
    }
    least = min(least, key);
  }
  atomicMin(&s.lo, least);
  __syncthreads();
  const uint32_t lowest = s.lo;
  __syncthreads();
  if (threadIdx.x == 0) s.hi = lowest;
  __syncthreads();
  if (found) s.hi = at;  // equal keys alone
  __syncthreads();
  const uint32_t got = s.hi;
  __syncthreads();
  return got;
}

// The least kept key from a row's list of at most KEYS
template <typename S, typename R>
INLINE uint32_t least_of_list(S& s, const RowState& state, const RowPlan& plan,
                                  const Wants& want, const R& row) {
  const int n = plan.n;
  for (int i = threadIdx.x; i < (n + 3) / 4 * 4; i += S::WG) {
    const uint32_t key = i < n ? state.list[i] : 0;
    s.key[i] = key;
    s.key_mass[i] = i < n && want.by_p ? units(row.weight(key2f(key))) : 0;
  }
  __syncthreads();
  uint32_t lo = 0xffffffffu, hi = 0;
  if (n > RANKED) {
    if (threadIdx.x == 0) {
      s.lo = lo;
      s.hi = hi;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += S::WG) {
      lo = min(lo, s.key[i]);
      hi = max(hi, s.key[i]);
    }
    atomicMin(&s.lo, lo);
    atomicMax(&s.hi, hi);
    __syncthreads();
    lo = s.lo;
    hi = s.hi;
    __syncthreads();
  }
  auto each_key = [&](auto f) {
    for (int i = threadIdx.x; i < n; i += S::WG) f(s.key[i]);
  };
  auto find = [&](auto by_mass, double above, double target) {
    constexpr bool BY_MASS = decltype(by_mass)::value;
    return n <= RANKED ? rank_keys<BY_MASS>(s, n, above, target)
                       : split_keys<BY_MASS>(s, row, lo, hi, above, target, each_key);
  };
  if (!want.by_k) return find(std::true_type(), plan.above, plan.target);
  const uint32_t kmin = find(std::false_type(), plan.above, plan.target);
  if (!want.by_p) return kmin;
  double kept = 0.0;  // the list has all that the first threshold keeps
  for (int i = threadIdx.x; i < n; i += S::WG)
    if (s.key[i] >= kmin) kept += s.key_mass[i] * UNIT;
  const double target = (double)want.p * (float)block_total(s, kept);
  if (target <= 0.0) return max(kmin, f2key(row.m));
  return max(kmin, find(std::true_type(), 0.0, target));
}

// ---- a row by one workgroup; of rows in CHUNKS the thresholds, and those rows that are left to it
template <typename T, typename F, bool CHUNKS>
__global__ __launch_bounds__(F::WG) void sample_fullvocab_kernel(const SampleArgs a,
                                                                 RowState* states) {
  constexpr int WG = F::WG, TILE = F::TILE;
  __shared__ Shared<F> s;
  const int n_row = blockIdx.x, t = threadIdx.x;
  const Wants want = wants_of(a, n_row);
  const int V = a.V;
  Row<T, WG> row = row_of<T, WG>(a, n_row);
  if (CHUNKS) {
    RowState& state = states[n_row];
    const RowPlan plan = state.plan;
    if (want.greedy || plan.mode == NO_LIST) return;
    if (!left_whole(plan)) {
      row.m = plan.m;
      const uint32_t least = least_of_list(s, state, plan, want, row);
      if (t == 0) state.plan.kmin = least;
      return;
    }
  }
  const int stride = (V + STRIPES - 1) / STRIPES;

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
  block_max(s, mx, best, odd);
  const bool plain = !odd;
  row.m = mx;
  if (want.greedy) {
    if (t == 0) a.out[n_row] = best < V ? best : 0;
    return;
  }

  // ---- top-k, then top-p: kept = {key >= kmin}
  const float p = want.p;
  const bool by_k = want.by_k, by_p = want.by_p;
  uint32_t kmin = 0;
  if (by_k) kmin = boundary<false>(s, row, want.k, 0.0, plain);
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
  draw(s, a, row, n_row, kmin, mine);
}

template <typename T>
static void launch(const SampleArgs& a, void* work, int chunks, hipStream_t stream) {
  using Small = Form<256, 16>;
  using Large = Form<1024, 64>;
  RowState* const states = (RowState*)work;
  const int grid = a.B * chunks;
  if (chunks) {
    chunk_max_kernel<T><<<grid, 256, 0, stream>>>(a, states, chunks);
    chunk_histogram_kernel<T><<<grid, 256, 0, stream>>>(a, states, chunks);
    chunk_keys_kernel<T><<<grid, 256, 0, stream>>>(a, states, chunks);
    sample_fullvocab_kernel<T, Large, true><<<a.B, Large::WG, 0, stream>>>(a, states);
    chunk_sums_kernel<T><<<grid, 256, 0, stream>>>(a, states, chunks);
    draw_kernel<T><<<a.B, 256, 0, stream>>>(a, states);
  } else if (a.V <= 4096 || (a.V <= 8192 && a.B > 256)) {
    sample_fullvocab_kernel<T, Small, false><<<a.B, Small::WG, 0, stream>>>(a, states);
  } else {
    sample_fullvocab_kernel<T, Large, false><<<a.B, Large::WG, 0, stream>>>(a, states);
  }
}

// Chunks of a row, the more of them the fewer the rows; 0: a workgroup a row, which is faster from 100 rows
// on, for smaller vocabularies, and for greedy rows that would wait for the launches.  By a workgroup a
// row and in chunks, us, greedy, plain, top-p and all kinds in turns: 128256 tokens 1 row 19 38 81 38 and
// 17 29 54 29, 16 20 41 85 84 and 19 34 63 63, 64 22 42 89 88 and 24 42 78 77, 100 23 44 90 89 and 27 51
// 95 94, 190 25 48 94 91 and 38 73 129 123; 100000 16 17 42 79 78 and 19 33 61 62; 65536 8 12 25 53 52
// and 17 27 49 50; 50257 8 13 30 60 59 and 18 28 47 48; 32000 8 8 20 39 39 and 15 24 40 41.
extern "C" int sample_fullvocab_chunks(int B, int V) {
  return V < SPLIT_VOCAB || B > 64 ? 0 : B <= 16 ? 32 : 16;
}

// What sample_fullvocab with that many chunks works in
extern "C" int64_t sample_fullvocab_bytes(int B, int chunks) {
  return chunks ? (int64_t)B * sizeof(RowState) : 0;
}

extern "C" void launch_sample_fullvocab(int64_t* out, const void* logits, bool bf16,
                             const float* temps, const int64_t* top_ks,
                             const float* top_ps, const float* uniforms,
                             const uint8_t* mask, const int32_t* mask_map,
                             int B, int V, void* work, int chunks, hipStream_t stream) {
  const SampleArgs a = {out, logits, temps, top_ks, top_ps, uniforms, mask, mask_map, B, V};
  if (bf16)
    launch<bf16_t>(a, work, chunks, stream);
  else
    launch<float>(a, work, chunks, stream);
}
