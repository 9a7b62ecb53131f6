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
// Against the GEMM library (and the unit's own pass), us: 64 x 4096 x 14336 31 (41), 192 x 28672
// x 4096 SwiGLU 58 (67), 192 x 4096 x 14336 46 (103), 512 x 4096 x 14336 67 (91), 1739 x 28672 x
// 4096 SwiGLU 328 (417), 7664 x 28672 x 4096 SwiGLU 1259 (1376), 10000 x 4096 x 4096 244 (370).
#include <math.h>

#include "launch.h"
#include "linear_tile.h"

#define CUS 256
#define LDS_OF_A_CU 163840

struct LinearGrid {
  int tiles_m, tiles_n, band;
  int splits, each;  // parts of the inner dimension, chunks of one
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
    const int tiles = grid.tiles_m * grid.tiles_n, chunks = a.K >> 6;
    const int base = t / step * step, i = t - base;
    const int here = min(step, total - base), q = here >> 3, r = here & 7, xcd = i & 7;
    int id = base + (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (i >> 3);
    const int part = grid.splits > 1 ? id / tiles : 0;
    id -= part * tiles;
    const int per = grid.band * grid.tiles_n, b = id / per, rest = id - b * per;
    const int high = min(grid.band, grid.tiles_m - b * grid.band), column = rest / high;
    const int first = part * grid.each, last = min(chunks, first + grid.each);
    const int at = first + (int)(column * grid.apart >> 32);
    return {(b * grid.band + rest % high) * tm, a.M, column * tn, first, last, part, a.w, a.x, a.M,
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

template <int UNIT>
static void sum(const LinearArgs& a, const void* parts, int splits, hipStream_t stream) {
  const int each = (a.K / 64 + splits - 1) / splits;
  const int64_t outs = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU ? a.N / 2 : a.N;
  const int count = (a.K / 64 + each - 1) / each;
  auto kernel = linear_sum_kernel<UNIT>;
  kernel<<<dim3((a.M * outs / 8 + 255) / 256), 256, 0, stream>>>(a, (const float*)parts, count);
}

struct Tile {
  int fn, fm, ws, xs;
};
// an odd number of pairs of fragments cannot hold gates and ups
#define TILES(T) \
  T(8, 8, 3, 2) T(8, 7, 3, 2) T(8, 6, 3, 2) T(8, 5, 3, 3) T(8, 4, 3, 4) \
  T(4, 6, 4, 4) T(4, 4, 5, 5) T(4, 3, 5, 5) T(4, 2, 3, 3) T(4, 1, 4, 4)
#define PLAIN_TILES(T) T(6, 4, 4, 4) T(2, 2, 5, 5) T(2, 1, 6, 6)
#define SIZES(fn, fm, ws, xs) {fn, fm, ws, xs},
static const Tile tiles[] = {TILES(SIZES) PLAIN_TILES(SIZES)};
static constexpr int GLU_TILES = 10;

static constexpr int TILE_COUNT = sizeof(tiles) / sizeof(Tile);

extern "C" bool linear_fits(int tile, bool glu) {
  return tile >= 0 && tile < (glu ? GLU_TILES : TILE_COUNT);
}

// The tile and the parts that are expected to be the fastest, in us: the chunks of the busiest
// CU, by its matrix cores or its LDS, beside the memory's time.  Fitted to 286 sizes of 8 to
// 10000 rows, 2048 to 128256 outputs and 768 to 14336 inner elements; what it chooses is on
// average 1% slower than the best of all tiles and parts, 12 to 19% where it is worst (64 x 4096 x
// 4096: 16.4, best 13.8).
extern "C" void linear_choice(int M, int N, int K, int unit, int* tile, int* splits) {
  static const int parts[] = {1, 2, 3, 4, 6, 8, 12, 16};
  const bool glu = unit == LINEAR_SWIGLU || unit == LINEAR_GLU;
  const int chunks = K / 64;
  double best = 0;
  *tile = -1;
  for (int i = 0; i < TILE_COUNT; ++i) {
    const Tile& t = tiles[i];
    if (t.fm > 1 && (t.fm - 1) * 32 >= M) continue;  // rows of nothing
    const int64_t grid = ((int64_t)M + 32 * t.fm - 1) / (32 * t.fm) *
                         (((int64_t)N + 32 * t.fn - 1) / (32 * t.fn));
    const double step = fmax(0.015 * t.fn * t.fm, 0.053 * (t.fn + t.fm));
    for (int s : parts) {
      if (s == 1 && glu && i >= GLU_TILES) continue;
      if (s > 1 && (chunks < 4 * s || M > 2600 || grid * s > 4 * CUS)) break;
      const int each = (chunks + s - 1) / s;
      const int64_t works = grid * ((chunks + each - 1) / each);
      const double busiest =
          (double)((works + CUS - 1) / CUS) * (each * step + 0.08 * t.fn * t.fm + 0.57);
      const double sums = s > 1 ? 8.0 * s * M * N : 2.0 * M * N;
      const double memory = (2.0 * N * K + 2.0 * M * K + sums) / 6.4e6;
      const double us =
          sqrt(busiest * busiest + memory * memory) +
          (s > 1 ? (unit == LINEAR_PARTS ? 0.5 : 4.3) + sums / 21.7e6 : 0);
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
#define LAUNCH_PLAIN(n, m, ws, xs)        \
  LAUNCH_AS(n, m, ws, xs, LINEAR_PLAIN)   \
  LAUNCH_AS(n, m, ws, xs, LINEAR_BIAS)    \
  LAUNCH_AS(n, m, ws, xs, LINEAR_PARTS)
#define LAUNCH(n, m, ws, xs)              \
  LAUNCH_PLAIN(n, m, ws, xs)              \
  LAUNCH_AS(n, m, ws, xs, LINEAR_SWIGLU)  \
  LAUNCH_AS(n, m, ws, xs, LINEAR_GLU)
  TILES(LAUNCH)
  PLAIN_TILES(LAUNCH_PLAIN)
  if (splits > 1 && unit != LINEAR_PARTS) {
    a.out = args->out;
    unit == LINEAR_PLAIN    ? sum<LINEAR_PLAIN>(a, parts, splits, stream)
    : unit == LINEAR_BIAS   ? sum<LINEAR_BIAS>(a, parts, splits, stream)
    : unit == LINEAR_SWIGLU ? sum<LINEAR_SWIGLU>(a, parts, splits, stream)
                            : sum<LINEAR_GLU>(a, parts, splits, stream);
  }
}
