// y = x w^T for more rows than step_linear.hip's (gfx950), with a bias or the gated unit of the
// two halves of y, which then needs no pass of its own.
//
// A workgroup of 4 waves owns a tile of 32 FN outputs and 32 FM rows, a wave a quarter of it;
// products 16x16x32 with the weights as the first operand, whose rows are taken in such an order
// that a lane ends with 8 neighbouring outputs of a row.  K goes in chunks of 64, a cache line
// a row, straight from memory to LDS (addresses swizzled at the source), in rings of WS chunks
// of w and XS of x.  Per chunk and wave two steps of FN FM products, among them the reads of the
// fragments of the next step and the loads of chunks ahead, and one barrier, an eighth into the
// second step: by then the chunk is read and the next one has landed.  The workgroups stay for
// all their tiles, and the loads run ahead over the end of a tile; works are in runs of an XCD,
// bands of up to 8 tiles of rows beside each other.  Few tiles take the inner dimension in
// parts, whose sums meet in a second launch, in their order, in fp32.
//
// Bound by the matrix cores and the card's power from about a thousand rows on (256 x 256 tiles:
// 1.77 GHz, 78% of the cycles in products), by reading the weights below.  Which of the orders
// matters most, 8131 x 4096 x 14336, us: 32x32x16 products 767 (at 1.75 GHz: they take more
// power for the same work), 16x16x32 in the compiler's order 890, with the reads and loads fixed
// among them 663, the reads done at three quarters of a step 652.  Stores of whole lines past
// the caches: 8131 x 28672 x 4096 1335 to 1299.
//
// Against the GEMM library (and the unit's own pass), us: 64 x 4096 x 14336 29 (43), 192 x 28672
// x 4096 SwiGLU 56 (67), 192 x 4096 x 14336 41 (104), 512 x 4096 x 14336 68 (91), 1739 x 28672 x
// 4096 SwiGLU 315 (422), 7664 x 28672 x 4096 SwiGLU 1278 (1397), 10000 x 4096 x 4096 242 (361),
// 15675 x 28672 x 4096 SwiGLU 2538 (2765), 1.45 PFLOP/s.
#include <math.h>

#include "launch.h"
#include "linear_tile.h"

#define CUS 256
#define LDS_OF_A_CU 163840

// n / by for n below 2^31 as a product (Granlund and Montgomery, 1994).  A division is about 30
// instructions one after another, and a launch waited for four times five of them ahead of its
// first and its last loads: 2048 x 2048 of 40 rows 8.8 us and now 8.3, 13 x 4096 x 4096 9.4 and 9.0, 61 x
// 6144 x 4096 15.6 and 15.4; by divisions of 64 bits one more each took 2 to 3 us.
struct Over {
  unsigned by, mul, shift;
};
static Over over(unsigned by) {
  unsigned shift = 0;
  while ((1ull << shift) < by) ++shift;
  return {by, (unsigned)(((1ull << 32) * ((1ull << shift) - by)) / by + 1), shift};
}
DEV int operator/(int n, const Over& d) {
  return (int)((__umulhi((unsigned)n, d.mul) + (unsigned)n) >> d.shift);
}

struct LinearGrid {
  int tiles_m, tiles_n, band;
  int splits, each;  // parts of the inner dimension, chunks of one
  Over step, tiles, per, high, low;  // workgroups, tiles, those of a band, rows of one, of the last
  uint64_t apart;    // chunks from where a tile begins to where its neighbour does, times 2^32
};

struct LinearWork {
  static constexpr bool ANY_WIDTH = false;
  const LinearArgs& a;
  const LinearGrid& grid;
  int tn, tm;  // outputs and rows of a tile
  int start, step, total;

  DEV int next(int t) const { return t + step < total ? t + step : t; }
  DEV int64_t x_row(const LinearSpot&, int m) const { return m; }
  DEV int64_t out_row(const LinearSpot&, int m) const { return m; }
  // XCDs have runs of a round's works, in bands of up to 8 tiles of rows beside each other
  DEV LinearSpot spot(int t) const {
    const int chunks = a.K >> 6, base = t / grid.step * step, i = t - base;
    const int here = min(step, total - base), q = here >> 3, r = here & 7, xcd = i & 7;
    int id = base + (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (i >> 3);
    const int part = grid.splits > 1 ? id / grid.tiles : 0;
    id -= part * (int)grid.tiles.by;
    const int b = id / grid.per, rest = id - b * (int)grid.per.by;
    const Over& high = (b + 1) * grid.band <= grid.tiles_m ? grid.high : grid.low;
    const int column = rest / high;
    const int first = part * grid.each, last = min(chunks, first + grid.each);
    const int at = first + (int)(column * grid.apart >> 32);
    return {(b * grid.band + rest - column * (int)high.by) * tm, a.M, column * tn, first, last, part, a.w, a.x, a.M,
            0, at};
  }
};

template <int FN, int FM, int WS, int XS, int UNIT, bool ONCE>
__global__ __launch_bounds__(256, 1) void linear_kernel(const LinearArgs a, const LinearGrid grid) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ char lds[];
  constexpr bool GLU = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU;
  const LinearWork work = {a, grid, GLU ? 16 * FN : 32 * FN, 32 * FM, (int)blockIdx.x,
                           (int)gridDim.x, grid.tiles_m * grid.tiles_n * grid.splits};
  linear_tiles<FN, FM, WS, XS, UNIT, ONCE>(a, work, lds);
#endif
}

// The parts' sums, in their order, through the unit: 8 outputs a thread
template <int UNIT>
__global__ __launch_bounds__(256) void linear_sum_kernel(const LinearArgs a, const float* parts,
                                                         const int splits) {
  constexpr bool GLU = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU;
  const int outs = GLU ? a.N / 2 : a.N, per_row = outs >> 3;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)a.M * per_row) return;
  const int64_t m = i / per_row;
  const int o = (int)(i - m * per_row) * 8;
  const float* from = parts + m * a.N + o;
  f32x4_v y[GLU ? 4 : 2] = {};
  for (int s = 0; s < splits; ++s, from += (int64_t)a.M * a.N) {
    y[0] += ((const f32x4_v*)from)[0];
    y[1] += ((const f32x4_v*)from)[1];
    if (GLU) {
      y[2 * GLU] += ((const f32x4_v*)(from + outs))[0];
      y[3 * GLU] += ((const f32x4_v*)(from + outs))[1];
    }
  }
  bf16x8_v v, b;
  if (UNIT == LINEAR_BIAS) b = *(const bf16x8_v*)((const __bf16*)a.bias + o);
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    float sum = y[r >> 2][r & 3];
    if (UNIT == LINEAR_BIAS) sum += (float)b[r];
    if (GLU) sum = unit_of<UNIT>(a, sum, y[(2 + (r >> 2)) * GLU][r & 3]);
    v[r] = (__bf16)sum;
  }
  *(bf16x8_v*)((__bf16*)a.out + m * a.out_stride + o) = v;
}

template <int FN, int FM, int WS, int XS, int UNIT>
static void launch(const LinearArgs& a, int splits, hipStream_t stream) {
  constexpr int TN = 32 * FN, TM = 32 * FM, LDS = 128 * (WS * TN + XS * TM);
  constexpr bool GLU = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU;
  static_assert(LDS <= LDS_OF_A_CU);
  if constexpr (!(GLU && FN % 4)) {  // linear_fits()
    allow_lds<linear_kernel<FN, FM, WS, XS, UNIT, false>>(LDS);
    allow_lds<linear_kernel<FN, FM, WS, XS, UNIT, true>>(LDS);
    const int outs = GLU ? a.N / 2 : a.N, per = GLU ? TN / 2 : TN, chunks = a.K / 64;
    LinearGrid g;
    g.tiles_m = (a.M + TM - 1) / TM;
    g.tiles_n = (outs + per - 1) / per;
    const int bands = (g.tiles_m + 7) / 8;
    g.band = (g.tiles_m + bands - 1) / bands;
    g.each = (chunks + splits - 1) / splits;
    g.splits = (chunks + g.each - 1) / g.each;
    const int total = g.tiles_m * g.tiles_n * g.splits, fit = CUS * (LDS_OF_A_CU / LDS);
    const int workgroups = total < fit ? total : fit;
    g.step = over(workgroups);
    g.tiles = over(g.tiles_m * g.tiles_n);
    g.per = over(g.band * g.tiles_n);
    g.high = over(g.band);
    g.low = over(g.tiles_m % g.band ? g.tiles_m % g.band : g.band);
    // One tile of rows reads the weights once: past the caches, us: 13 x 28672 x 4096 SwiGLU 48.6 to
    // 44.3, 13 x 12288 x 4096 22.5 to 20.9, 61 x 128256 x 4096 209 to 193, 13 x 17792 x 2048 19.4 to
    // 18.6; weights of 33 MB are not worth it, 13 x 2048 x 8192 12.9 and 13.9
    const bool once = g.tiles_m == 1 && (int64_t)a.N * a.K >= 32 << 20;
    // Rows of a power of two lie 4 KB and more apart, so that their columns are in a few of the memory's
    // channels, all of which are busy only if tiles are at different columns.  us, before and now: 61 x
    // 28672 x 4096 SwiGLU 50.9 and 42.5, 13 x 28672 x 4096 47.0 and 39.5, 13 x 12288 x 4096 20.6 and
    // 18.3, 61 x 20480 x 4096 44.5 and 42.1, 190 x 128256 x 4096 231 and 192; at K = 5120 or 3584 the
    // same as before.  Weights in rows of 64 elements more give no less, for more memory; an eighth
    // of K apart by XCD 1 to 5% less, by twos or fours of tiles nothing.  Parts are apart by themselves: 61 x
    // 6144 x 4096 in 4 parts 14.0, in turns 14.9.
    g.apart = once && g.splits == 1 ? ((uint64_t)chunks << 32) / g.tiles_n : 0;
    auto kernel = once ? linear_kernel<FN, FM, WS, XS, UNIT, true>
                       : linear_kernel<FN, FM, WS, XS, UNIT, false>;
    kernel<<<dim3(workgroups), 256, LDS, stream>>>(a, g);
  }
}

template <int UNIT>
static void sum(const LinearArgs& a, const void* parts, int splits, hipStream_t stream) {
  const int each = (a.K / 64 + splits - 1) / splits;
  const int64_t outs = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU ? a.N / 2 : a.N;
  const int count = (a.K / 64 + each - 1) / each;
  auto kernel = linear_sum_kernel<UNIT>;
  kernel<<<dim3((a.M * outs / 8 + 255) / 256), 256, 0, stream>>>(a, (const float*)parts, count);
}

// step: us of a chunk
struct Tile {
  int fn, fm, ws, xs;
  double step;
};
// The rings' depths: 61 x 28672 x 4096 SwiGLU by 128 x 64 with 3 chunks of both 42.5, with 4 40.0;
// 190 rows of it by 128 x 192 with 4 59.7, with 3 57.2
#define TILES(T)                                                                             \
  T(8, 8, 3, 2, 1.142) T(8, 7, 3, 2, 1.034) T(8, 6, 3, 2, 0.891) T(8, 5, 3, 3, 0.802)        \
  T(8, 4, 3, 4, 0.753) T(4, 6, 3, 3, 0.614) T(4, 4, 5, 5, 0.55) T(4, 3, 5, 5, 0.446)         \
  T(4, 2, 4, 4, 0.393) T(4, 1, 4, 4, 0.34) T(6, 4, 4, 4, 0.674) T(2, 2, 5, 5, 0.234)         \
  T(2, 1, 6, 6, 0.185) T(4, 5, 4, 3, 0.561)
#define SIZES(fn, fm, ws, xs, step) {fn, fm, ws, xs, step},
static const Tile tiles[] = {TILES(SIZES)};
static constexpr int TILE_COUNT = sizeof(tiles) / sizeof(Tile);

// an odd number of pairs of fragments cannot hold gates and ups
extern "C" bool linear_fits(int tile, bool glu) {
  return tile >= 0 && tile < TILE_COUNT && !(glu && tiles[tile].fn % 4);
}

// (a^1.36 + b^1.36)^(1 / 1.36), by the ratio of a to b: a table's 256 steps of it, which are at most 1e-4
// off, take a tenth of three powers
struct Together {
  double of[258];
  Together() {
    for (int i = 0; i < 258; ++i) of[i] = pow(1 + pow(i / 256.0, 1.36), 1 / 1.36);
  }
  double operator()(double a, double b) const {
    const double high = a > b ? a : b, at = (a > b ? b : a) / high * 256;
    const int i = (int)at;
    return high * (of[i] + (at - i) * (of[i + 1] - of[i]));
  }
};
static const Together together;

// The tile and the parts that are expected to be the fastest, in us: the chunks of the busiest
// CU beside the memory's time.  A chunk takes as long as its rows take to be loaded, so that a tile of
// rows which is not full takes less.  Fitted to 2200 products of 5 to 2100 rows by 32 sizes of weights,
// 1024 to 37888 outputs and 1280 to 13824 inner elements, some with the norm that adds up their parts.
// What it chooses is on average 1.1% slower than the best of all tiles and parts, 7% and more in one of
// 20, 20% where it is worst; fitted to one half of the weights 1.4 and 1.7% on the other half, and 1.0% on
// 396 products into the rotation that it was not fitted to.  A model with one time for a tile's chunks, full
// or not, and a term for what tiles read again: 1.7%, 28% where it is worst, as it took tiles of 64 x 64 that
// are whole in the inner dimension, and few large ones in parts.  us by it and now: 190 x 5120 x 5120 into
// the norm 28.9 and 22.6, 777 x 4096 x 4096 40.3 and 32.2, 512 x 2048 x 8192 36.4 and 30.2.
// Above 2100 rows, where the matrix cores and the card's power bound a tile, steps are by the fragments,
// as fitted to 8 to 10000 rows.  A choice by a table there, where it was another one, was 0.6% slower on average
// of 110 products of 2101 to 16384 rows, 5.7% at worst and 5.2% faster at best: 2500 x 28672 x 4096 SwiGLU
// 444 us by fragments and 469, 7664 x 16384 x 2048 399 and 414, 10000 x 6144 x 4096 371 and 387, but 13000 x
// 28672 x 4096 2178 and 2129; 15675 rows of it 2562 and 2548, 2584 and 2580.
// It is asked for every launch and takes 0.1 to 0.7 us, 0.3 to 3.8 with powers for each of up to 154 pairs.
extern "C" void linear_choice(int M, int N, int K, int unit, int* tile, int* splits) {
  static const int parts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16};
  constexpr int PARTS = sizeof(parts) / sizeof(int);
  const bool glu = unit == LINEAR_SWIGLU || unit == LINEAR_GLU, few = M <= 2100;
  const int chunks = K / 64, most = M > 2600 ? 1 : chunks / 4;
  const double rows = 2.0 * M * K, weights = 2.0 * N * K, outs = (double)M * N;
  int each[PARTS], count[PARTS], n = 1;
  each[0] = chunks, count[0] = 1;
  for (; n < PARTS && parts[n] <= most; ++n) {
    each[n] = (chunks + parts[n] - 1) / parts[n];
    count[n] = (chunks + each[n] - 1) / each[n];
  }
  double best = 0;
  *tile = -1;
  for (int i = 0; i < TILE_COUNT; ++i) {
    const Tile& t = tiles[i];
    if (t.fm > 1 && (t.fm - 1) * 32 >= M) continue;  // rows of nothing
    const unsigned high = (M - 1u) / (32 * t.fm) + 1, wide = (N - 1u) / (32 * t.fn) + 1;
    const int64_t grid = (int64_t)high * wide;
    const double fragments = t.fn * t.fm;
    const double loaded = (32.0 * t.fn + (double)M / high) / (32 * (t.fn + t.fm));
    const double step = few ? t.step * loaded : fmax(0.015 * fragments, 0.053 * (t.fn + t.fm));
    const double ends = few ? 0.125 * fragments + 0.887 : 0.08 * fragments + 0.57;
    for (int j = 0; j < n; ++j) {
      const int s = parts[j];
      if (s == 1 && !linear_fits(i, glu)) continue;
      if (s > 1 && grid * s > 4 * CUS) break;
      const int64_t works = grid * count[j];
      const double busiest = (double)((works + CUS - 1) / CUS) * (each[j] * step + ends);
      const double sums = (s > 1 ? 8.0 * count[j] : glu && few ? 1.0 : 2.0) * outs;
      const double memory = (weights + rows + sums) / (few ? 6.1e6 : 6.4e6);
      const double rest =
          s == 1 ? 0
          : few  ? (unit == LINEAR_PARTS ? 0 : 4.0) + sums / 27e6  // 3.5 in a graph, 4.3 outside
                 : (unit == LINEAR_PARTS ? 0.5 : 4.3) + sums / 21.7e6;
      // both together take less than their sum, and no less than by squares
      const double squares = busiest * busiest + memory * memory, room = best - rest;
      if (*tile >= 0 && (room <= 0 || squares >= room * room)) continue;
      const double us = rest + (few ? together(busiest, memory) : sqrt(squares));
      if (*tile >= 0 && us >= best) continue;
      best = us;
      *tile = i;
      *splits = s;
    }
  }
}

extern "C" void launch_linear(const LinearArgs* args, int unit, int tile, int splits, void* parts,
                              hipStream_t stream) {
  const Tile t = tiles[tile];
  LinearArgs a = *args;
  int kind = unit;
  if (splits > 1) {
    kind = LINEAR_PARTS;
    a.out = parts;
  } else if (unit == LINEAR_PARTS) {
    kind = LINEAR_PLAIN;
  }
#define LAUNCH_AS(n, m, ws_, xs_, u)                                       \
  if (kind == u && t.fn == n && t.fm == m && t.ws == ws_ && t.xs == xs_)   \
    launch<n, m, ws_, xs_, u>(a, splits, stream);
#define LAUNCH(n, m, ws, xs, step)        \
  LAUNCH_AS(n, m, ws, xs, LINEAR_PLAIN)   \
  LAUNCH_AS(n, m, ws, xs, LINEAR_BIAS)    \
  LAUNCH_AS(n, m, ws, xs, LINEAR_PARTS)   \
  LAUNCH_AS(n, m, ws, xs, LINEAR_SWIGLU)  \
  LAUNCH_AS(n, m, ws, xs, LINEAR_GLU)
  TILES(LAUNCH)
  if (splits > 1 && unit != LINEAR_PARTS) {
    a.out = args->out;
    unit == LINEAR_PLAIN    ? sum<LINEAR_PLAIN>(a, parts, splits, stream)
    : unit == LINEAR_BIAS   ? sum<LINEAR_BIAS>(a, parts, splits, stream)
    : unit == LINEAR_SWIGLU ? sum<LINEAR_SWIGLU>(a, parts, splits, stream)
                            : sum<LINEAR_GLU>(a, parts, splits, stream);
  }
}
