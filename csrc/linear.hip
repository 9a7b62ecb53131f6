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
// Against the GEMM library (and the unit's own pass), us: 64 x 4096 x 14336 30 (53), 192 x 28672
// x 4096 SwiGLU 69 (72), 192 x 4096 x 14336 42 (111), 512 x 4096 x 14336 70 (98), 1739 x 28672 x
// 4096 SwiGLU 329 (422), 7664 x 28672 x 4096 SwiGLU 1296 (1458), 10000 x 4096 x 4096 251 (361).
#include <math.h>

#include <type_traits>

#include "common_t.h"
#include "gated_act.h"
#include "linear.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;

#define CUS 256
#define LDS_OF_A_CU 163840

struct LinearGrid {
  int tiles_m, tiles_n, band;
  int splits, each;  // parts of the inner dimension, chunks of one
};

// The gated unit of two sums, both rounded first, as they are between two passes
template <int UNIT>
DEV float unit_of(const LinearArgs& a, float gate, float up) {
  gate = (float)(__bf16)gate;
  up = (float)(__bf16)up;
  if (UNIT == LINEAR_SWIGLU) return gate * __builtin_amdgcn_rcpf(1.f + __expf(-gate)) * up;
  return clamped_glu_f(gate, up, a.limit, a.alpha, a.offset, a.cubic);
}

// Fragments of a wave along the outputs (FN) and the rows (FM); XS: chunks of x in LDS.
template <int FN, int FM, int WS, int XS, int UNIT>
__global__ __launch_bounds__(256, 1) void linear_kernel(const LinearArgs a, const LinearGrid grid) {
#ifdef __HIP_DEVICE_COMPILE__  // the host knows no buffer resources
  extern __shared__ char lds[];
  constexpr bool GLU = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU;
  constexpr int TN = 32 * FN, TM = 32 * FM;    // rows of w and of x of a tile
  constexpr int LW = FN, LX = FM;              // a wave's loads of a chunk, 8 rows each
  constexpr int SW = TN * 128, SX = TM * 128;  // a chunk's bytes
  constexpr int NM = FN * FM;
  // loads behind a chunk's last one when it is waited for
  constexpr int BEHIND = XS < WS ? LW + (XS - 2) * (LW + LX) : (WS - 2) * (LW + LX);
  static_assert(BEHIND < 64 && WS >= 3 && XS >= 2);
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wid & 1, wm = wid >> 1;
  const int c = lane & 15, g = lane >> 4;
  const int outs = GLU ? a.N / 2 : a.N;
  const int tiles = grid.tiles_m * grid.tiles_n, total = tiles * grid.splits, nwg = gridDim.x;
  const int chunks = a.K >> 6;

  // part of the inner dimension, first row and output of work t
  auto place = [&](int t, int& part, int& m0, int& o0) {
    const int base = t / nwg * nwg, i = t - base;
    const int here = min(nwg, total - base), q = here >> 3, r = here & 7, xcd = i & 7;
    int id = base + (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (i >> 3);
    part = UNIT == LINEAR_PARTS ? id / tiles : 0;
    id -= part * tiles;
    const int per = grid.band * grid.tiles_n, b = id / per, rest = id - b * per;
    const int high = min(grid.band, grid.tiles_m - b * grid.band);
    m0 = (b * grid.band + rest % high) * TM;
    o0 = rest / high * (GLU ? TN / 2 : TN);
  };

  auto buffer = [](const void* p, int64_t rows, int64_t stride, int64_t row) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(((rows - 1) * stride + row) * 2),
                                             0x00020000);
  };
  const auto bw = buffer(a.w, a.N, a.w_stride, a.K), bx = buffer(a.x, a.M, a.x_stride, a.K);
  const int slot = ((lane & 7) ^ (lane >> 3)) * 16;
  int vw[LW], vx[LX];  // this lane's rows
  auto first_chunk = [&](int part) { return UNIT == LINEAR_PARTS ? part * grid.each : 0; };
  auto last_chunk = [&](int part) {
    return UNIT == LINEAR_PARTS ? min(chunks, (part + 1) * grid.each) : chunks;
  };
  // cursors of the loads: work, chunk, its last one, place in LDS; past the last work its
  // chunks again
  int tw = blockIdx.x, cw, ew, sw = 0, tx = blockIdx.x, cx, ex, sx = 0;
  auto aim_w = [&](int t) {
    int part, m0, o0;
    place(t, part, m0, o0);
    cw = first_chunk(part);
    ew = last_chunk(part);
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      // in such an order that a lane's sums are of 8 neighbours
      const int p = (wid * LW + i) * 8 + (lane >> 3), f = p >> 4, k = p & 15;
      const int in = 8 * (k >> 2) + 4 * (f & 1) + (k & 3);
      int o = min(o0 + (GLU ? f >> 2 : f >> 1) * 32 + in, outs - 1);
      if (GLU && (f & 2)) o += outs;
      vw[i] = (int)(o * a.w_stride) * 2 + slot;
    }
  };
  auto aim_x = [&](int t) {
    int part, m0, o0;
    place(t, part, m0, o0);
    cx = first_chunk(part);
    ex = last_chunk(part);
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int p = (wid * LX + i) * 8 + (lane >> 3);
      vx[i] = (int)(min(m0 + p, a.M - 1) * a.x_stride) * 2 + slot;
    }
  };
  auto load_w = [&](int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(bw, (lds_char*)(lds + sw + (wid * LW + i) * 1024), 16,
                                             vw[i], cw * 128, 0, 0);
  };
  auto load_x = [&](int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        bx, (lds_char*)(lds + WS * SW + sx + (wid * LX + i) * 1024), 16, vx[i], cx * 128, 0, 0);
  };
  auto next_w = [&]() {
    sw = sw == (WS - 1) * SW ? 0 : sw + SW;
    if (++cw == ew) {
      if (tw + nwg < total) tw += nwg;
      aim_w(tw);
    }
  };
  auto next_x = [&]() {
    sx = sx == (XS - 1) * SX ? 0 : sx + SX;
    if (++cx == ex) {
      if (tx + nwg < total) tx += nwg;
      aim_x(tx);
    }
  };

  // fragments: row c of 16, 8 inner elements of step s (32 of the chunk's 64)
  const int pw = (wn * FN * 16 + c) * 128, px = WS * SW + (wm * FM * 16 + c) * 128;
  const int at[2] = {(g ^ (c & 7)) * 16, ((4 + g) ^ (c & 7)) * 16};
  bf16x8_v fw[2][FN], fx[2][FM];
  int rw = 0, rx = 0;  // the chunk that is read
  const char *qw, *qx;
  auto look = [&](int s) {
    qw = lds + (rw + pw + at[s]);
    qx = lds + (rx + px + at[s]);
  };
  // the n-th fragment of FN + FM, as the products need them
  auto read = [&](int set, int n) {
    constexpr int BOTH = FN < FM ? FN : FM;
    const int i = n < 2 * BOTH ? n >> 1 : n - BOTH;
    if (n < 2 * BOTH ? !(n & 1) : FN > FM)
      fw[set][i] = *(const bf16x8_v*)(qw + i * 2048);
    else
      fx[set][i] = *(const bf16x8_v*)(qx + i * 2048);
  };
  f32x4_v acc[FN][FM];
  // products FROM .. TO - 1 of a set of fragments by growing corners (the first ones need the
  // first fragments), among them the other set's R reads, done at three quarters, and L loads
  auto multiply = [&](auto first, auto fixed_set, auto from, auto to, auto reads, auto loads,
                      auto&& load) {
    constexpr int set = decltype(fixed_set)::value, F = decltype(from)::value;
    constexpr int T = decltype(to)::value, R = decltype(reads)::value, L = decltype(loads)::value;
    int n = 0, r = 0, l = 0;
#pragma unroll
    for (int k = 0; k < (FN > FM ? FN : FM); ++k)
#pragma unroll
      for (int q = 0; q <= 2 * k; ++q) {
        const int i = q & 1 ? k : q >> 1, j = q & 1 ? q >> 1 : k;
        if (i >= FN || j >= FM) continue;
        if (n >= F && n < T) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              fw[set][i], fx[set][j], decltype(first)::value ? f32x4_v{} : acc[i][j], 0, 0, 0);
          bool cut = false;
          while (r < R && 3 * r * (T - F) <= 4 * (n - F) * R) read(set ^ 1, r++), cut = true;
          while (l < L && (2 * l + 1) * (T - F) <= 2 * (n - F) * L) load(l++), cut = true;
          if (cut) __builtin_amdgcn_sched_barrier(0);
        }
        ++n;
      }
    while (r < R) read(set ^ 1, r++);
    while (l < L) load(l++);
    __builtin_amdgcn_sched_barrier(0);
  };

  aim_w(tw);
  aim_x(tx);
#pragma unroll
  for (int k = 0; k < (WS > XS ? WS - 1 : XS); ++k) {
    if (k < WS - 1) {
#pragma unroll
      for (int i = 0; i < LW; ++i) load_w(i);
      next_w();
    }
    if (k < XS) {
#pragma unroll
      for (int i = 0; i < LX; ++i) load_x(i);
      next_x();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  look(0);
#pragma unroll
  for (int i = 0; i < FN + FM; ++i) read(0, i);

  for (int t = blockIdx.x; t < total; t += nwg) {
    int part, m0, o0;
    place(t, part, m0, o0);
    auto chunk = [&](auto first) {
      typedef std::integral_constant<int, 0> I0;
      typedef std::integral_constant<int, 1> I1;
      typedef std::integral_constant<int, NM / 8> Ahead;
      typedef std::integral_constant<int, NM> All;
      typedef std::integral_constant<int, FN + FM> Reads;
      look(1);
      multiply(first, I0(), I0(), All(), Reads(), std::integral_constant<int, LW>(), load_w);
      next_w();
      multiply(std::false_type(), I1(), I0(), Ahead(), I0(), I0(), load_x);
      // this chunk is read, the next one has landed, for every wave after the barrier; what
      // may be under way are the loads behind the next chunk's
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      rw = rw == (WS - 1) * SW ? 0 : rw + SW;
      rx = rx == (XS - 1) * SX ? 0 : rx + SX;
      look(0);
      multiply(std::false_type(), I1(), Ahead(), All(), Reads(), std::integral_constant<int, LX>(),
               load_x);
      next_x();
    };
    chunk(std::true_type());
    for (int k = last_chunk(part) - first_chunk(part); k > 1; --k) chunk(std::false_type());

    // sums r of fragments i (and i + 1) and j: row c of 16, outputs 8 g + r (and 4 + r) of 32
    constexpr int GROUP = GLU ? 4 : 2;  // fragments of 32 outputs
    if (UNIT == LINEAR_PARTS) {
      float* const sums = (float*)a.out + part * (int64_t)a.M * a.N;
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const int m = m0 + (wm * FM + j) * 16 + c;
        if (m >= a.M) continue;
#pragma unroll
        for (int i = 0; i < FN; i += 2) {
          const int o = o0 + (wn * FN + i) * 16 + 8 * g;
          if (o >= outs) continue;
          f32x4_v* const to = (f32x4_v*)(sums + m * (int64_t)a.N + o);
          to[0] = acc[i][j];
          to[1] = acc[i + 1][j];
        }
      }
      continue;
    }
    auto eight = [&](int i, int j, int o) {
      bf16x8_v v, b;
      if (UNIT == LINEAR_BIAS) b = *(const bf16x8_v*)((const __bf16*)a.bias + min(o, outs - 8));
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        float y = acc[i + (r >> 2)][j][r & 3];
        if (GLU) {
          y = unit_of<UNIT>(a, y, acc[i + (GLU ? 2 : 0) + (r >> 2)][j][r & 3]);
        } else if (UNIT == LINEAR_BIAS) {
          y += (float)b[r];
        }
        v[r] = (__bf16)y;
      }
      return __builtin_bit_cast(u32x4_v, v);
    };
    __bf16* const out = (__bf16*)a.out;
    const bool low = c < 8;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + (wm * FM + j) * 16;
#pragma unroll
      for (int i = 0; i < FN; i += 2 * GROUP) {
        const int o = o0 + (wn * (FN / GROUP) + i / GROUP) * 32 + 8 * g;
        const u32x4_v p = eight(i, j, o);
        if (i + GROUP < FN) {
          // whole lines: 8 rows of 64 outputs a store, by lanes 8 apart
          const u32x4_v q = eight(i + GROUP < FN ? i + GROUP : i, j, o + 32);
          u32x4_v upper, lower;
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const unsigned other =
                __builtin_amdgcn_update_dpp(0, low ? q[d] : p[d], 0x128, 0xf, 0xf, false);
            upper[d] = low ? p[d] : other;
            lower[d] = low ? other : q[d];
          }
          const int oo = low ? o : o + 32, mm = m + (c & 7);
          __bf16* const to = out + mm * a.out_stride + oo;
          if (oo < outs) {
            if (mm < a.M) __builtin_nontemporal_store(upper, (u32x4_v*)to);
            if (mm + 8 < a.M) __builtin_nontemporal_store(lower, (u32x4_v*)(to + 8 * a.out_stride));
          }
        } else if (m + c < a.M && o < outs) {
          __builtin_nontemporal_store(p, (u32x4_v*)(out + (m + c) * a.out_stride + o));
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end
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
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)linear_kernel<FN, FM, WS, XS, UNIT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    attr_set = true;
  }
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
  auto kernel = linear_kernel<FN, FM, WS, XS, UNIT>;
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
          sqrt(busiest * busiest + memory * memory) + (s > 1 ? 4.3 + sums / 21.7e6 : 0);
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
  if (splits > 1) {
    a.out = args->out;
    unit == LINEAR_PLAIN    ? sum<LINEAR_PLAIN>(a, parts, splits, stream)
    : unit == LINEAR_BIAS   ? sum<LINEAR_BIAS>(a, parts, splits, stream)
    : unit == LINEAR_SWIGLU ? sum<LINEAR_SWIGLU>(a, parts, splits, stream)
                            : sum<LINEAR_GLU>(a, parts, splits, stream);
  }
}
