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
// thread a stripe: one after another in fp32 without a threshold (all CUTS are false), by fours in
// fp32 and those in 64 bits with one.
//
// Greedy rows of whole units by one workgroup, and those with a threshold, take another way, by
// units (below), and this one where that does not fit.  190 rows of 128256 in fp32 by this one,
// other logits each time, whole calls: 25 us greedy, 49 plain, 79 top-k, 95 top-p, 135 both (26,
// 58, 97, 168 and 238 with calls of functions, which take a row and LDS by reference: their loads
// and atomics then go by unknown memory and wait for both kinds).  Floating masses instead of whole
// ones in the histogram took as long, a shared list of the bucket 25 us more.
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

#define HELD 16      // units of a thread in registers
#define STREAM 2     // others asked for ahead
#define UNIT_KEYS 4096
#define UNIT_BUCKETS 512
#define PARTS 128    // of a bucket
#define PARTS_OF_BUCKET (1 << 19)  // of a column: from there on its count
#define PER_OCTAVE 16
#define PER_LOGIT 8  // likewise, of a top-k
// beyond it more keys are within the masses' error than the list takes: normal logits 3000 at 0.99 of
// 128256 and 4400 of 152064
// (from 0.999 on the masses' error reaches all of the row)
#define MOST_P(V) fminf(1.f - (V) * 7.6e-8f, 0.9985f)

// the number before the -3.4e38 that a row's largest logit is at least: what is equal to that is found
#define BELOW -0x1.ff933ep127f

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

// Tokens of a stripe; with a threshold in whole fours of the row
template <bool CUTS = true>
__device__ __forceinline__ int stripe_tokens(int V) {
  const int n = (V + STRIPES - 1) / STRIPES;
  return CUTS ? (n + 3) & ~3 : n;
}
// Weights of a row with a threshold are added up by fours, those in 64 bits
template <bool CUTS>
using SumOf = std::conditional_t<CUTS, double, float>;
__device__ __forceinline__ float sum_of_four(float a, float b, float c, float d) {
  return (a + c) + (b + d);
}
// The token of a four whose weight takes ``before`` beyond target, or the last one of any weight
__device__ __forceinline__ int token_of_four(const float* w, double before, double target) {
  int last = 0;
  for (int e = 0; e < 4; ++e) {
    if (w[e] > 0.f) last = e;
    if ((before += w[e]) > target) return e;
  }
  return last;
}

// Threads of a workgroup, and tokens of a stripe that are summed at a time.  With 1024 threads and
// 160 KB a CU has one row, and each step of a row ends in a wait for 16 waves: small vocabularies
// take 256 threads and 61 KB.  1024 and 256 threads, us: 512 rows of 600 greedy 10.7 and 5.7, plain
// 24.9 and 10.9, 16 rows of 4096 plain 14.2 and 9.8, top-p 29 and 24.  From there on only where
// the rows are more than the CUs: 512 rows of 8192 plain 30.8 and 15.6, but 16 rows top-p with a
// mask 32 and 39.
template <int THREADS, int TOKENS>
struct Form {
  static constexpr int WG = THREADS, WAVES = WG / 64, TILE = TOKENS;
  static constexpr bool LISTS = WG == 1024;  // rows by units, and lists of rows in chunks
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
    // a row's by units, by lanes, so that no two lanes of a wave meet: count, and parts of a bucket
    alignas(16) uint32_t column[F::LISTS ? UNIT_BUCKETS : 1][64];
    struct {
      alignas(16) uint32_t key[F::LISTS ? UNIT_KEYS : 1];  // of a row in chunks, or by units
      unsigned long long key_mass[F::LISTS ? UNIT_KEYS : 1];
      int key_wave[F::LISTS ? UNIT_KEYS : 1];
      alignas(16) uint32_t sub_key[F::LISTS ? RANKED + 4 : 1];
      unsigned long long sub_mass[F::LISTS ? RANKED + 4 : 1];
      unsigned long long wave_units[F::WAVES];
      // of the drawn wave
      double unit_sum[F::LISTS ? MOST_VOCAB / 4 / F::WAVES + 64 : 1];
      double turn_sum[F::LISTS ? MOST_VOCAB / 256 / F::WAVES + 1 : 1];
    };
  };
  float stripe[STRIPES], cdf[STRIPES + 1];  // of a row without a threshold
  double wave[F::WAVES];
  float red[F::WAVES];
  int red_i[F::WAVES], red_odd[F::WAVES];
  int n, pick, finite, listed;
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
  float m, invT, scale;  // the largest logit, 1 / temperature, that in octaves

  template <bool CUTS = true>
  __device__ float weight(float v) const {
    return CUTS ? __builtin_amdgcn_exp2f((v - m) * scale) : __expf((v - m) * invT);
  }

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

// Sum over the threads before, and of all
template <typename S>
INLINE double scan_block(S& s, double v, double* all) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double upto = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double w = __shfl_up(upto, off, 64);
    if (lane >= off) upto += w;
  }
  if (lane == 63) s.wave[wid] = upto;
  __syncthreads();
  double before = 0.0, total = 0.0;
#pragma unroll 2
  for (int i = 0; i < S::WAVES; ++i) {
    if (i == wid) before = total;
    total += s.wave[i];
  }
  __syncthreads();
  *all = total;
  return before + upto - v;
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
  const float temp = a.temps[n], invT = temp <= 0.f ? 1.f : 1.f / temp;
  return {(const T*)a.logits + (int64_t)n * a.V,
          masked ? a.mask + (int64_t)a.mask_map[n] * a.V : nullptr, a.V, 0.f, invT,
          invT * 1.44269504f};
}

// A stripe's weights of a tile; WIDE: all of them on their way from LDS at once also for sums in 64
// bits, where a thread has the registers (rows in chunks: 16 x 128256 top-k 7.6 us by halves, 7.0)
template <bool CUTS, int TILE, bool WIDE = false>
INLINE void add_tile(const float* tile, SumOf<CUTS>& sum) {
  constexpr int FOURS = !CUTS || WIDE || TILE < 32 ? TILE / 4 : 8;
#pragma unroll 1
  for (int j0 = 0; j0 < TILE / 4; j0 += FOURS) {
    float4 w[FOURS];
#pragma unroll
    for (int j = 0; j < FOURS; ++j) w[j] = *(const float4*)(tile + 4 * (j0 + j));
#pragma unroll
    for (int j = 0; j < FOURS; ++j) {
      if constexpr (CUTS)
        sum += sum_of_four(w[j].x, w[j].y, w[j].z, w[j].w);
      else
        sum = sum + w[j].x + w[j].y + w[j].z + w[j].w;
    }
  }
}

// ---- inverse-CDF draw in token-id order from the stripes' sums, ``mine`` of the t-th thread's.
// Without a threshold sums are in fp32, in order, by one thread; with one in 64 bits, where a scan
// is the faster one: 1 x 128256 top-k in chunks 43.5 us in order, 41.2 by the scan.  Compiled apart,
// since what asks for the kind at each weight, or has both kinds' sums in 64 bits, is slower: plain
// rows by a workgroup a row 60 us for 190 x 128256, 49 so; 64 x 4104 18.2 and 13.9.
template <bool CUTS, typename S, typename R>
INLINE void draw(S& s, const SampleArgs& a, const R& row, int n_row, uint32_t kmin,
                     SumOf<CUTS> mine) {
  using Sum = SumOf<CUTS>;
  constexpr int WG = S::WG;
  const int t = threadIdx.x, V = row.V, stride = stripe_tokens<CUTS>(V);
  constexpr int STEP = 32;  // one thread's LDS reads in flight
  Sum ahead = 0, target = 0;
  int n = -1;
  if constexpr (CUTS) {
    if (t == 0) {
      s.pick = -1;
      s.n = STRIPES;
    }
    const double own = t < STRIPES ? mine : 0.0;
    double all;
    const double before = scan_block(s, own, &all);
    target = (double)a.uniforms[n_row] * all;
    if (own > 0.0 && before + own > target) atomicMin(&s.n, t);
    __syncthreads();
    n = s.n;
    if (t == n) s.above = before;
    __syncthreads();
    ahead = s.above;
    if (n == STRIPES) n = -1;
  } else {
    if (t < STRIPES) s.stripe[t] = mine;
    if (t == 0) s.pick = s.n = -1;
    __syncthreads();
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
    target = a.uniforms[n_row] * s.cdf[STRIPES];
    // exactly one stripe satisfies prefix <= target < prefix + mine
    // (mine > 0 guaranteed for the owner since the CDF strictly increases
    // across it); fp edge cases fall through to the fallback below
    if (t < STRIPES && mine > 0.f && s.cdf[t] <= target && target < s.cdf[t + 1]) s.n = t;
    __syncthreads();
    n = s.n;
    __syncthreads();
    if (n >= 0) ahead = s.cdf[n];
  }
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
          w = row.template weight<CUTS>(v);
          last = i0 + j;
        }
      }
      buf[j] = w;
    }
    if (last >= 0) atomicMax(&s.pick, last);
    __syncthreads();
    if (t == 0) {
      Sum cum = ahead;
      int first = -1;
      for (int j = 0; j < here && first < 0; j += STEP) {
        float w[STEP], fours[STEP / 4];
        Sum upto = cum;
#pragma unroll
        for (int e = 0; e < STEP; e += 4) {
          *(float4*)(w + e) = *(const float4*)(buf + j + e);
          if constexpr (CUTS) {
            fours[e / 4] = sum_of_four(w[e], w[e + 1], w[e + 2], w[e + 3]);
            upto += fours[e / 4];
          }
        }
        if constexpr (!CUTS) {
#pragma unroll
          for (int e = 0; e < STEP; ++e) upto += w[e];
        }
        if (!(upto <= target)) {  // the same sums again: weights are not negative
          if constexpr (CUTS) {
#pragma unroll
            for (int g = 0; g < STEP / 4; ++g) {
              if (first < 0 && cum + fours[g] > target)
                first = 4 * g + token_of_four(w + 4 * g, cum, target);
              cum += fours[g];
            }
          } else {
            for (int e = 0; e < STEP && first < 0; ++e)
              if ((cum += buf[j + e]) > target) first = e;
          }
        }
        cum = upto;
        if (first >= 0) s.pick = i0 + j + first;
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

// A row's state between the launches.  What many workgroups add to or read begins at a cache line, 16 x
// 128256 top-k: histogram 8.2 us otherwise and 7.7, keys 13.7 and 12.9
struct RowState {
  RowPlan plan;
  double rest[MOST_CHUNKS];
  float chunk_max[MOST_CHUNKS];
  int chunk_best[MOST_CHUNKS], chunk_odd[MOST_CHUNKS];
  double stripe[STRIPES];
  alignas(128) uint32_t list[KEYS];
  alignas(128) uint32_t count[FIRST];
  alignas(128) unsigned long long mass[FIRST];
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
template <bool CUTS = true>
__device__ __forceinline__ Chunk chunk_of(const SampleArgs& a, int chunks) {
  Chunk c;
  c.row = blockIdx.x / chunks;
  c.at = blockIdx.x - c.row * chunks;
  c.stride = stripe_tokens<CUTS>(a.V);
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

template <bool CUTS, typename T>
INLINE void chunk_sums(ChunkShared& s, const SampleArgs& a, const Chunk& c, const Row<T, 256>& row,
                       const RowPlan& plan, RowState& state) {
  constexpr int TILE = ChunkForm::TILE;
  const int t = threadIdx.x;
  const uint32_t kmin = plan.kmin;
  // stripes' weights by all threads, 64 tokens of each at a time, added up by a thread a stripe
  const int r = t / TILE, col = t % TILE;
  constexpr int ROWS = 256 / TILE, MOST = STRIPES / LEAST_CHUNKS / ROWS;
  const float least = key2f(kmin);
  const bool by_value = kmin == 0 || (least == least && least != 0.f);
  const float from = kmin == 0 ? -INFINITY : least;
  float ahead[MOST];
  SumOf<CUTS> mine = 0;
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
      tile[k * ROWS + r][col] = in ? row.template weight<CUTS>(ahead[k]) : 0.f;
    }
    if (j0 + TILE < c.stride) fetch(j0 + TILE);
    __syncthreads();  // the other tile is added up before it is written again
    if (t < c.stripes) add_tile<CUTS, TILE, true>(tile[t], mine);
  }
  if (t < c.stripes) state.stripe[c.at * c.stripes + t] = mine;
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_sums_kernel(const SampleArgs a, RowState* states,
                                                         const int chunks) {
  __shared__ ChunkShared s;
  const int n_row = blockIdx.x / chunks;
  const Wants want = wants_of(a, n_row);
  if (want.greedy) return;
  Row<T, 256> row = row_of<T, 256>(a, n_row);
  RowState& state = states[n_row];
  const RowPlan plan = state.plan;
  row.m = plan.m;
  if (left_whole(plan)) return;
  if (want.by_k || want.by_p)
    chunk_sums<true>(s, a, chunk_of<true>(a, chunks), row, plan, state);
  else
    chunk_sums<false>(s, a, chunk_of<false>(a, chunks), row, plan, state);
}

struct DrawShared : ChunkForm {
  alignas(16) float buffer[MOST_VOCAB / STRIPES + 64];
  float stripe[STRIPES], cdf[STRIPES + 1];
  double wave[WAVES], above;
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
  const Wants want = wants_of(a, n_row);
  if (want.by_k || want.by_p)
    draw<true>(s, a, row, n_row, plan.kmin, state.stripe[threadIdx.x]);
  else
    draw<false>(s, a, row, n_row, plan.kmin, (float)state.stripe[threadIdx.x]);
}

// The key of a list at which the sum from the top, with what is ``above``, reaches target, the
// least one if rounding lets none do so.  A thread compares its key with all others, which takes
// 33 ns a key; the two rounds of split_keys take about 12 us whatever the list: RANKED keys.
template <bool BY_MASS, typename S>
INLINE uint32_t rank_keys(S& s, const uint32_t* keys, const unsigned long long* masses, int n,
                          double above, double target) {
  if (threadIdx.x == 0) s.lo = 0xffffffffu;
  __syncthreads();
  uint32_t least = 0xffffffffu, at = 0;
  bool found = false;
  for (int i = threadIdx.x; i < n; i += S::WG) {
    const uint32_t key = keys[i];
    unsigned long long higher = 0, same = 0;
    for (int j = 0; j < n; j += 4) {
      const u32x4 k = *(const u32x4*)&keys[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // the units behind the last key are 0
        const unsigned long long w = BY_MASS ? masses[j + e] : j + e < n;
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
INLINE uint32_t least_of_list(S& s, const uint32_t* list, int n, double above, double target,
                              const Wants& want, const R& row) {
  for (int i = threadIdx.x; i < (n + 3) / 4 * 4; i += S::WG) {
    const uint32_t key = i < n ? list[i] : 0;
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
  auto find = [&, first = lo, last = hi](auto by_mass, double above, double target) {
    uint32_t lo = first, hi = last;
    constexpr bool BY_MASS = decltype(by_mass)::value;
    if (n <= RANKED) return rank_keys<BY_MASS>(s, s.key, s.key_mass, n, above, target);
    if constexpr (S::LISTS) {
      // a round of split_keys(), after which its bucket has few: 500 keys 6 us, its two rounds 12
      const int shift = hi - lo < SPLIT ? 0 : 32 - __builtin_clz(hi - lo) - 10;
      for (int i = threadIdx.x; i < SPLIT; i += S::WG) s.mass[i] = 0;
      if (threadIdx.x == 0) s.n = 0;
      __syncthreads();
      for (int i = threadIdx.x; i < n; i += S::WG)
        atomicAdd(&s.mass[(hi - s.key[i]) >> shift], BY_MASS ? s.key_mass[i] : 1ull);
      __syncthreads();
      const double unit = BY_MASS ? UNIT : 1.0;
      double all, mine = s.mass[threadIdx.x] * unit;
      const double before = above + scan_block(s, mine, &all);
      if (before < target && before + mine >= target) {
        s.above = before;
        s.n = 1 + (int)threadIdx.x;
      }
      __syncthreads();
      const int bucket = s.n - 1;
      const double sub_above = s.above;
      __syncthreads();
      if (threadIdx.x == 0) s.n = 0;
      __syncthreads();
      if (bucket >= 0) {
        for (int i = threadIdx.x; i < n; i += S::WG)
          if ((int)((hi - s.key[i]) >> shift) == bucket) {
            const int at = atomicAdd(&s.n, 1);
            if (at < RANKED) {
              s.sub_key[at] = s.key[i];
              s.sub_mass[at] = s.key_mass[i];
            }
          }
        __syncthreads();
        const int few = s.n;
        // many of one key, as logits of 16 bits have them, need neither ranks nor a split: 16 x 128256 in
        // chunks, logits of a twentieth and a top-p of 0.9, 75 us by ranks, 62 so
        hi -= (uint32_t)bucket << shift;
        lo = max(lo, hi - ((1u << shift) - 1));
        const uint32_t one = s.sub_key[0];
        int others = 0;
        for (int i = threadIdx.x; i < n; i += S::WG)
          others |= s.key[i] >= lo && s.key[i] <= hi && s.key[i] != one;
        if (!__syncthreads_or(others)) return one;
        if (few <= RANKED) {
          if (threadIdx.x < 4) {
            s.sub_key[few + threadIdx.x] = 0;
            s.sub_mass[few + threadIdx.x] = 0;
          }
          __syncthreads();
          return rank_keys<BY_MASS>(s, s.sub_key, s.sub_mass, few, sub_above, target);
        }
        above = sub_above;
      }
    }
    return split_keys<BY_MASS>(s, row, lo, hi, above, target, each_key);
  };
  if (!want.by_k) return find(std::true_type(), above, target);
  const uint32_t kmin = find(std::false_type(), above, target);
  if (!want.by_p) return kmin;
  double kept = 0.0;  // the list has all that the first threshold keeps
  for (int i = threadIdx.x; i < n; i += S::WG)
    if (s.key[i] >= kmin) kept += s.key_mass[i] * UNIT;
  const double of_kept = (double)want.p * (float)block_total(s, kept);
  if (of_kept <= 0.0) return max(kmin, f2key(row.m));
  return max(kmin, find(std::true_type(), 0.0, of_kept));
}

// inverse-CDF draw in token-id order over the kept set, {key >= kmin}
template <bool CUTS, typename S, typename R>
INLINE void sum_and_draw(S& s, const SampleArgs& a, const R& row, int n_row, uint32_t kmin,
                         bool plain) {
  constexpr int WG = S::WG, TILE = S::TILE;
  const int t = threadIdx.x, V = row.V, stride = stripe_tokens<CUTS>(V);
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
  SumOf<CUTS> mine = 0;
  fetch(0);
  for (int j0 = 0; j0 < stride; j0 += TILE) {
    float(*tile)[TILE + 4] = s.tile[j0 / TILE % 2];
    const bool by_values = by_value && plain && !row.mask && j0 + TILE <= stride;
    if (by_values && even) {
#pragma unroll
      for (int k = 0; k < PER; ++k)
        tile[k * ROWS + r][c] = ahead[k] >= from ? row.template weight<CUTS>(ahead[k]) : 0.f;
    } else if (by_values) {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const bool in = ahead[k] >= from && k * ROWS * stride + j0 + i_first < V;
        tile[k * ROWS + r][c] = in ? row.template weight<CUTS>(ahead[k]) : 0.f;
      }
    } else {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int i = k * ROWS * stride + j0 + i_first;
        const bool in = j0 + c < stride && i < V && f2key(ahead[k]) >= kmin &&
                        !(row.mask && !row.mask[i]);
        tile[k * ROWS + r][c] = in ? row.template weight<CUTS>(ahead[k]) : 0.f;
      }
    }
    if (j0 + TILE < stride) fetch(j0 + TILE);
    __syncthreads();  // the other tile is added up before it is written again
    if (t < STRIPES) add_tile<CUTS, TILE>(tile[t], mine);
  }
  draw<CUTS>(s, a, row, n_row, kmin, mine);
}

// ---- a row by one workgroup, in as many passes over it as its thresholds call for
template <typename T, typename S>
INLINE void whole_row(S& s, const SampleArgs& a, const Wants& want, Row<T, S::WG>& row, int n_row) {
  const int t = threadIdx.x, V = a.V;

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

  if (by_k || by_p)
    sum_and_draw<true>(s, a, row, n_row, kmin, plain);
  else
    sum_and_draw<false>(s, a, row, n_row, kmin, plain);
}

// ---- a row by one workgroup, by units of 16 bytes
//
// A wave owns consecutive units, 64 a turn, and keeps the first HELD turns in registers (half of a row
// of 128256 in fp32); the rest comes from memory in every pass.  An instruction an element is about 1 us a
// pass for 16 waves, and reading a row 16 to 19, so both count:
//   1 the largest logit, by three-way maxima; a greedy row's is found again in its unit
//   2 for a threshold, a histogram over the distance to it, 16 buckets an octave of the weight or finer:
//     per bucket and lane the count and the sum of the distances within it, in one word, so that no
//     two lanes of a wave meet (64-bit atomics on one table took 75 us instead of 10).  A bucket's
//     mass is known to 4e-4 from both, so which buckets the boundary can be in, and no weight is made
//   3 the weights above those buckets in a thread's own sum in 64 bits, the keys in them into a list, from
//     which the least kept key follows exactly
// The draw goes to the wave that has the target, then to its turn, a unit, a token, in token-id order.
// 190 rows of 128256 in fp32, whole_row() and this, us: greedy 25 and 23, top-k 81 and 56, top-p 96 and
// 77, both 136 and 62, top-p 0.9 at a temperature of 6.4 100 and 79; bf16 22 and 14, 71 and 47, 93 and
// 64, 119 and 52; 32000 in fp32 11 and 10, 37 and 27, 43 and 36, 59 and 33; 70% allowed by a mask 59
// and 33, 173 and 79, 221 and 96, 310 and 85.  Plain rows took 33 instead of 49, but their draws are by
// sums in fp32, in order, and one in 50 was another one by these sums: they stay whole_row()'s.  With
// more registers HELD they spill, and a build with spills drew wrong tokens; 4 units ahead instead of 2
// as long.
// A row that this does not fit is whole_row()'s: one of no threshold that is not greedy, of no whole
// units, logits that are no numbers or all alike, a boundary among more keys than the list has (from
// -inf among logits that no mask has out, buckets do not narrow) or beyond the last bucket, a top-p
// beyond MOST_P.
template <typename T, bool MASKED>
struct Units {
  static constexpr int N = 16 / sizeof(T);
  const char* x;
  const uint8_t* mask;      // or null, MASKED
  int count, first, turns;  // units of the row, the wave's first one and its turns of 64

  DEV static float at(const u32x4& v, int e) {
    const uint32_t bits = N == 4 ? v[e & 3] : (e & 1) ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16;
    return __uint_as_float(bits);
  }
  // the last one in place of units beyond it
  DEV u32x4 load(int u) const { return *(const u32x4*)(x + (uint32_t)min(u, count - 1) * 16u); }
  // units beyond the last one, and tokens that are not allowed, are logits of no weight; ``some``:
  // there may be units beyond
  DEV void clear(u32x4& v, int u, bool some) const {
    if (some && u >= count) {
#pragma unroll
      for (int d = 0; d < 4; ++d) v[d] = N == 4 ? 0xff800000u : 0xff80ff80u;
    }
    if (MASKED && mask) {
      const uint8_t* const allowed = mask + min(u, count - 1) * N;
#pragma unroll
      for (int e = 0; e < N; ++e) {
        if (allowed[e]) continue;
        if (N == 4)
          v[e & 3] = 0xff800000u;
        else
          v[e >> 1] = (e & 1) ? (v[e >> 1] & 0xffffu) | 0xff800000u : (v[e >> 1] & 0xffff0000u) | 0xff80u;
      }
    }
  }
  // without a branch, behind which a load would have to be waited for
  DEV u32x4 turn(int a) const { return load(first + a * 64 + (int)(threadIdx.x & 63)); }
  DEV void clear_turn(u32x4& v, int a) const {
    const int u = first + a * 64;
    clear(v, u + (int)(threadIdx.x & 63), u + 64 > count);
  }
  // f(unit, turn) of all turns, the held ones from registers.  The first time units beyond the last one
  // are that one again
  template <bool FIRST_TIME, typename F>
  DEV void each(u32x4 (&held)[HELD], F f) const {
    u32x4 next[STREAM];
#pragma unroll
    for (int g = 0; g < STREAM; ++g) next[g] = turn(HELD + g);
#pragma unroll
    for (int a = 0; a < HELD; ++a)
      if (a < turns) {
        if (FIRST_TIME && MASKED) clear_turn(held[a], a);
        f(held[a], a);
        if (FIRST_TIME && !MASKED) clear_turn(held[a], a);
      }
    for (int a = HELD; a < turns; a += STREAM) {
#pragma unroll
      for (int g = 0; g < STREAM; ++g) {
        u32x4 v = next[g];
        next[g] = turn(a + STREAM + g);
        if (a + g < turns) {
          if (!FIRST_TIME || MASKED) clear_turn(v, a + g);
          f(v, a + g);
        }
      }
    }
  }
};

DEV float max3(float a, float b, float c) {
  asm("v_max3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(b), "v"(c));
  return a;
}
DEV float min3(float a, float b, float c) {
  asm("v_min3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(b), "v"(c));
  return a;
}

// The least of the threads' logits
template <typename S>
INLINE float block_least(S& s, float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, 64));
  if ((threadIdx.x & 63) == 0) s.red[threadIdx.x >> 6] = v;
  __syncthreads();
#pragma unroll 4
  for (int w = 0; w < S::WAVES; ++w) v = fminf(v, s.red[w]);
  __syncthreads();
  return v;
}

// The first lane whose sum with those before it exceeds target, and the sum before it; 64: none
INLINE int first_above(double v, double target, double* before) {
  const int lane = threadIdx.x & 63;
  double upto = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double w = __shfl_up(upto, off, 64);
    if (lane >= off) upto += w;
  }
  const unsigned long long above = __ballot(v > 0.0 && upto > target);
  if (!above) return 64;
  const int at = __builtin_ctzll(above);
  *before = __shfl(upto - v, at, 64);
  return at;
}

template <typename T, bool MASKED, typename S>
INLINE bool row_by_units(S& s, const SampleArgs& a, const Wants& want, Row<T, S::WG>& row, int n_row) {
  using U = Units<T, MASKED>;
  constexpr int N = U::N, WAVES = S::WAVES;
  const int t = threadIdx.x, lane = t & 63, wid = __builtin_amdgcn_readfirstlane(t >> 6), V = a.V;
  if (V % N || (uintptr_t)row.x % 16) return false;
  const bool cuts = want.by_k || want.by_p;
  // with both the list has all that the top-k keeps, and what else its last bucket has: 190 x 128256
  // top-k 7000 and top-p 152 us, in 3 passes ahead of whole_row() 200
  if (!want.greedy && want.by_p &&
      !(want.p > 0.f && (want.by_k ? want.k <= UNIT_KEYS / 8 * 7 : want.p <= MOST_P(V))))
    return false;
  U units_of;
  units_of.x = (const char*)row.x;
  units_of.mask = row.mask;
  units_of.count = V / N;
  units_of.turns = (units_of.count + 64 * WAVES - 1) / (64 * WAVES);
  units_of.first = wid * units_of.turns * 64;
  // ---- 1
  float mx = BELOW, least = INFINITY;
  int best = 1 << 30, odd = 0;
  if (want.greedy) {
    // loads beyond a short row's end take longer than the passes save: 64 x 8192 7.6 us, 7.0 by
    // whole_row(); 64 x 16384 7.5 and 7.7
    if (units_of.turns < 4) return false;
    u32x4 held[HELD];
#pragma unroll
    for (int k = 0; k < HELD; ++k) held[k] = units_of.turn(k);
    units_of.template each<true>(held, [&](const u32x4& v, int k) {
      float y = BELOW;
#pragma unroll
      for (int e = 0; e < N; e += 2) y = max3(y, U::at(v, e), U::at(v, e + 1));
      if (y > mx) {
        mx = y;
        best = units_of.first + k * 64 + lane;
      }
    });
    block_max(s, mx, best, odd);
    if (t == 0) {
      int at = 0;
      if (best < units_of.count) {
        u32x4 v = units_of.load(best);
        units_of.clear(v, best, false);
#pragma unroll
        for (int e = N - 1; e >= 0; --e)
          if (U::at(v, e) == mx) at = best * N + e;
      }
      a.out[n_row] = at;
    }
    return true;
  }
  // plain rows turn back ahead of the loads (61 us and 49: 190 x 128256), which greedy rows have
  // their own of: with one set of them for all rows, and a return ahead of it, registers spill
  if (!cuts) return false;
  u32x4 held[HELD];
#pragma unroll
  for (int k = 0; k < HELD; ++k) held[k] = units_of.turn(k);
  if (t == 0) s.n = s.finite = s.listed = 0;
  for (int i = t; i < UNIT_BUCKETS * 16; i += S::WG) ((u32x4*)s.column)[i] = u32x4{};
  unsigned long long odd_lanes = 0;
  int finite = 0;  // of a masked row: the wave's logits above -inf
  units_of.template each<true>(held, [&](const u32x4& v, int) {
    if (MASKED && row.mask) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        const float x = U::at(v, e);
        const bool some = !(x == -INFINITY);
        mx = fmaxf(mx, x);
        least = fminf(least, some ? x : INFINITY);
        finite += __popcll(__ballot(some));
        odd_lanes |= __ballot(x != x);
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < N; e += 2) {
      const float x = U::at(v, e), y = U::at(v, e + 1);
      mx = max3(mx, x, y);
      least = min3(least, x, y);
      odd_lanes |= __ballot(__builtin_isunordered(x, y));
    }
  });
  odd = odd_lanes != 0;
  block_max(s, mx, best, odd);
  // top-k's buckets are of logits, so that no temperature takes the k-th beyond the last one
  const float per_octave = row.scale;
  float scale = want.by_k ? (float)PER_LOGIT / PER_OCTAVE : per_octave;
  // finer ones where the row does not reach the last one
  if (lane == 0) atomicAdd(&s.finite, finite);
  least = block_least(s, least);
  // a masked row of no more logits than its top-k keeps them all: no buckets.  190 x 128256 of 256 tokens,
  // top-k 2000: 57 us, 222 where the buckets were looked through for it before whole_row(), which takes
  // 187.  Likewise buckets span the allowed logits alone: normal ones times 0.05, top-k 78, 232 and 171
  const bool whole = MASKED && row.mask && want.by_k && s.finite <= want.k;
  if (!whole) {
    const float span = (mx - least) * scale, most = UNIT_BUCKETS / PER_OCTAVE - 2;
    if (!(span > 1e-20f)) return false;
    if (span < most) scale *= most / span;
    if (!(scale < 1e25f)) return false;
  }
  const float fine = scale * (PER_OCTAVE * PARTS), bucket_octaves = per_octave / scale / PER_OCTAVE;
  if (odd || !(mx > -1e37f && mx < INFINITY) || !(per_octave < 1e20f && per_octave > 1e-20f)) return false;
  row.m = mx;

  // ---- 2: the buckets lo .. hi - 1 that the boundary can be in
  int lo = 0, hi = 0;
  double k_above = 0.0;
  if (!whole) {
    uint32_t* const mine = &s.column[0][lane];
    units_of.template each<false>(held, [&](const u32x4& v, int) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        const float d = (mx - U::at(v, e)) * fine;
        if (d < (float)(UNIT_BUCKETS * PARTS)) {  // beyond 32 octaves all weigh less than the slack
          const uint32_t q = (uint32_t)d;
          atomicAdd(mine + q / PARTS * 64, (uint32_t)PARTS_OF_BUCKET | (q % PARTS));
        }
      }
    });
    if (t == 0) s.lo = s.hi = UNIT_BUCKETS;
    __syncthreads();
    // two threads a bucket
    static_assert(S::WG == 2 * UNIT_BUCKETS);
    static_assert(MOST_VOCAB / 64 * (PARTS - 1) < PARTS_OF_BUCKET, "a lane's parts stay below its count");
    static_assert((int64_t)MOST_VOCAB / 64 * PARTS_OF_BUCKET < 1ll << 32, "and its count in the word");
    const int b = t >> 1;
    uint32_t numbers = 0, parts = 0;
#pragma unroll 4
    for (int i = 0; i < 32; ++i) {
      const uint32_t h = s.column[b][(i + lane) % 32 + (t & 1) * 32];
      numbers += h / PARTS_OF_BUCKET;
      parts += h % PARTS_OF_BUCKET;
    }
    numbers += __shfl_xor(numbers, 1);
    parts += __shfl_xor(parts, 1);
    const double n = t & 1 ? 0.0 : (double)numbers;
    double after = 0.0, before = 0.0, all = 0.0;
    if (want.by_k) {
      // the bucket of the k-th; with both, all down to it are listed
      before = scan_block(s, n, &all);
      if (before < want.k && before + n >= want.k) {
        s.hi = b + 1;
        s.above = before;
      }
    } else {
      // the mean of a bucket's weights, in units of that at its edge, by the mean of the distances
      const double off =
          n > 0.0 ? ((double)parts / n + 0.5) * (0.6931471806 / PARTS) * bucket_octaves : 0.0;
      const double mass =
          n * (1.0 - off + 0.5 * off * off) * (double)__builtin_amdgcn_exp2f(b * -bucket_octaves);
      before = scan_block(s, mass, &all);
      after = before + mass;
      constexpr double SLACK = 5e-4;
      const double low = (double)want.p * all * (1 - SLACK), high = (double)want.p * all * (1 + SLACK);
      if (before * (1 + SLACK) < low && after * (1 + SLACK) >= low) s.lo = b;
      if (before * (1 - SLACK) < high && after * (1 - SLACK) >= high) s.hi = b + 1;
    }
    __syncthreads();
    hi = (int)s.hi;
    lo = want.by_p ? (want.by_k ? 0 : (int)s.lo) : hi - 1;
    k_above = want.by_k && !want.by_p ? s.above : 0.0;
    // what is beyond the last bucket is not told apart
    if (hi >= UNIT_BUCKETS || lo >= hi) return false;
    if (n > 0.0 && b >= lo && b < hi) atomicAdd(&s.listed, (int)numbers);
    __syncthreads();
    if (s.listed > UNIT_KEYS) return false;  // not after a pass that lists them, 30 us
  }

  // ---- 3
  // as the buckets are, whose scale differs by a power of two
  const float edge_lo = whole && !want.by_p ? -INFINITY : lo * (-1.f / PER_OCTAVE);
  const float edge_hi = whole ? -INFINITY : hi * (-1.f / PER_OCTAVE);
  // The masses that a top-p compares are added up weight by weight, so that the small ones count beside
  // a large one: by fours in fp32 a row's is off by up to 2^-25 of it.  190 x 128256 top-p 77 us, by
  // fours 73.  A top-k compares counts, and its sums are those of the draw alone
  const bool by_mass = !want.by_k;
  double kept = 0.0, all = 0.0;
  // not the differences of pass 2, which would be kept for it beside the logits
  float top = mx;
  asm volatile("" : "+v"(top));
  auto weigh = [&](float x) { return __builtin_amdgcn_exp2f((x - top) * per_octave); };
  units_of.template each<false>(held, [&](const u32x4& v, int) {
    float w[N], in[N];
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const float x = U::at(v, e), z = (x - top) * scale;
      w[e] = weigh(x);
      in[e] = z > edge_lo ? w[e] : 0.f;
      if (z > edge_hi && !(z > edge_lo)) {
        const int at = atomicAdd(&s.n, 1);
        if (at < UNIT_KEYS) {
          s.key[at] = f2key(x);
          s.key_wave[at] = wid;
        }
      }
    }
    if (by_mass) {
#pragma unroll
      for (int e = 0; e < N; ++e) {
        kept += (double)in[e];
        all += (double)w[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < N; e += 4)
        kept += (double)sum_of_four(in[e], in[e + 1], in[e + 2], in[e + 3]);
    }
  });
  uint32_t kmin = 0;
  if (t < WAVES) s.wave_units[t] = 0;
  if (!whole || want.by_p) {
    const double above = want.by_k ? k_above : block_total(s, kept);
    const double target = want.by_k ? want.k : (double)want.p * block_total(s, all);
    __syncthreads();
    const int n = s.n;
    if (n > UNIT_KEYS || n == 0 || !(above < target)) return false;
    kmin = least_of_list(s, s.key, n, above, target, want, row);
    // the least key of the list may be so because the list ends there
    double sum = 0.0;
    if (!want.by_k)
      for (int i = t; i < n; i += S::WG) sum += s.key_mass[i] * UNIT;
    if (!want.by_k && above + block_total(s, sum) < target) return false;
    for (int i = t; i < n; i += S::WG)
      if (s.key[i] >= kmin) atomicAdd(&s.wave_units[s.key_wave[i]], units(row.weight(key2f(s.key[i]))));
  }
  __syncthreads();

  // ---- the draw: the wave, then 64 units, a unit, a token
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) kept += __shfl_xor(kept, off, 64);
  if (lane == 0) s.wave[wid] = kept + s.wave_units[wid] * UNIT;
  __syncthreads();
  double total = 0.0;
#pragma unroll 2
  for (int i = 0; i < WAVES; ++i) total += s.wave[i];
  if (!(total > 0.0 && total < 1e30)) return false;
  const double target = (double)a.uniforms[n_row] * total;
  double before = 0.0;
  int drawn = -1, last = 0;
#pragma unroll 1
  for (int i = 0; i < WAVES && drawn < 0; ++i) {
    const double w = s.wave[i];
    if (w > 0.0) {
      last = i;
      if (before + w > target) drawn = i;
    }
    if (drawn < 0) before += w;
  }
  if (drawn < 0) {
    drawn = last;  // its last token
    before = -1e300;
  }
  const double rest = before > -1e299 ? target - before : 1e300;
  auto weights_of = [&](int u, float (&w)[N]) {
    u32x4 v = units_of.load(u);
    units_of.clear(v, u, true);
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const float x = U::at(v, e);
      w[e] = f2key(x) >= kmin ? weigh(x) : 0.f;
    }
  };
  const int first = drawn * units_of.turns * 64;
  for (int k = wid; k < units_of.turns; k += WAVES) {
    float w[N];
    weights_of(first + k * 64 + lane, w);
    double sum = 0.0;
#pragma unroll
    for (int e = 0; e < N; ++e) sum += (double)w[e];
    s.unit_sum[k * 64 + lane] = sum;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (lane == 0) s.turn_sum[k] = sum;
  }
  __syncthreads();
  if (wid) return true;
  double ahead = 0.0, at_turn = 0.0;
  const double mine = lane < units_of.turns ? s.turn_sum[lane] : 0.0;
  int k = first_above(mine, rest, &at_turn), u;
  const unsigned long long some = __ballot(mine > 0.0);
  bool end = k == 64;
  if (end) k = some ? 63 - __builtin_clzll(some) : 0;
  const double in_turn = s.unit_sum[k * 64 + lane];
  u = end ? 64 : first_above(in_turn, rest - at_turn, &ahead);
  const unsigned long long these = __ballot(in_turn > 0.0);
  if (u == 64) {
    end = true;
    u = these ? 63 - __builtin_clzll(these) : 0;
  }
  if (lane == 0) {
    float w[N];
    const int unit = first + k * 64 + u;
    weights_of(unit, w);
    double upto = at_turn + ahead;
    int pick = -1, last = 0;
#pragma unroll
    for (int e = 0; e < N; ++e) {
      upto += (double)w[e];
      if (w[e] > 0.f) last = e;
      if (pick < 0 && !end && w[e] > 0.f && upto > rest) pick = e;
    }
    a.out[n_row] = min(unit * N + (pick < 0 ? last : pick), V - 1);
  }
  return true;
}

// ---- a workgroup a row; of rows in CHUNKS the thresholds, and those rows that are left to it
template <typename T, typename F, bool CHUNKS, bool MASKED = true>
__global__ __launch_bounds__(F::WG) void sample_fullvocab_kernel(const SampleArgs a,
                                                                 RowState* states) {
  __shared__ Shared<F> s;
  const int n_row = blockIdx.x;
  const Wants want = wants_of(a, n_row);
  Row<T, F::WG> row = row_of<T, F::WG>(a, n_row);
  if constexpr (CHUNKS) {
    RowState& state = states[n_row];
    const RowPlan plan = state.plan;
    if (want.greedy || plan.mode == NO_LIST) return;
    if (!left_whole(plan)) {
      row.m = plan.m;
      const uint32_t least = least_of_list(s, state.list, plan.n, plan.above, plan.target, want, row);
      if (threadIdx.x == 0) state.plan.kmin = least;
      return;
    }
  } else if constexpr (F::LISTS) {
    if (row_by_units<T, MASKED>(s, a, want, row, n_row)) return;
  }
  whole_row<T>(s, a, want, row, n_row);
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
  } else if (a.mask && a.mask_map) {
    sample_fullvocab_kernel<T, Large, false><<<a.B, Large::WG, 0, stream>>>(a, states);
  } else {
    sample_fullvocab_kernel<T, Large, false, false><<<a.B, Large::WG, 0, stream>>>(a, states);
  }
}

// Chunks of a row, the more of them the fewer the rows; 0: a workgroup a row, which is faster from 65
// rows on and for smaller vocabularies.  By a workgroup a row and in chunks, us of fp32:
//                  greedy     plain      top-k      top-p      both       all kinds in turns
//   1 x 128256      8 17      37 27      40 40      52 51      46 47
//   16             10 19      40 32      42 45      59 59      48 52      58 58
//   32             10 19      41 34      43 50      60 65      49 57      60 63
//   64             11 22      41 39      43 59      61 73      50 66      60 70
//   100            13 28      42 53      45 86      62 103     51 93      61 81
//   16 x 65536      7 20      26 28      28 39      37 45      34 46      36 49
// So up to 64 rows it is plain rows, which go by whole_row(), that chunks are for; what rows want is known
// on the device alone.  A top-p of 0.999 takes 117 us in one workgroup and 139 in chunks, whose lists it
// does not fit either.
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
