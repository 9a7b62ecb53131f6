// The routed experts' products for many rows per expert (gfx950): a grouped GEMM over
// tiles of up to 256 rows of one expert.
//
// Rows come grouped by expert.  The first product gathers its token rows and applies the gated
// unit to its sums; the second reads the grouped rows in place and scatters its results to their
// (token, choice) entries.  A workgroup has one of linear_tile.h's tiles, of 256 rows of weights
// and of the height that its rows call for.  Where they stay for several tiles instead, the
// loads ahead wait for the next tile's rows and the shares are fixed: 10% slower.
//
// Bound by the matrix cores and the card's power for hundreds of rows an expert (59 and 52% of the
// cycles in products at 512, the rest the last round and the start of a tile), by the weights at
// 5 TB/s below.  32 experts of 4096 x 2560, 4 a token at random, both products, before (32x32x16
// products, 8 waves of 128 x 64, tiles of 256 rows or up to 320) and now, us: 128 tokens 452 and
// 416, 1024 538 and 428, 2048 669 and 612, 4093 1084 and 993, 8192 2009 and 1738; 16 of 2048 x
// 1536: 512 tokens 127 and 98, 2048 220 and 212, 4093 360 and 346, 8192 755 and 612.
#include "experts.h"
#include "launch.h"
#include "linear_tile.h"

#define LDS_BYTES 163840

// One tile
template <bool GLU>
struct ExpertWork {
  static constexpr bool ANY_WIDTH = !GLU;
  const ExpertsArgs& a;
  int row0, rows, o0;  // of the grouped rows
  const void* w;
  static constexpr int start = 0, step = 1, total = 1;

  DEV int next(int t) const { return t; }
  DEV LinearSpot spot(int) const {
    const __bf16* x = (const __bf16*)a.x + (GLU ? 0 : row0 * a.x_stride);
    return {0, rows, o0, 0, a.K >> 6, 0, w, x, GLU ? a.entries / a.top : rows, row0, 0};
  }
  DEV int64_t x_row(const LinearSpot& s, int m) const {
    return GLU ? a.perm[s.row0 + m] / a.top : m;
  }
  DEV int64_t out_row(const LinearSpot& s, int m) const {
    return GLU ? s.row0 + m : a.perm[s.row0 + m];
  }
};

template <bool GLU>
__global__ __launch_bounds__(256, 1) void experts_gemm_kernel(const ExpertsArgs a, const int tiles_n,
                                                              const int columns) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ char lds[];
  // The tiles come by their heights, the highest first; XCDs take blocks of 4 row tiles by up to
  // 5 columns in turns, so that all end with the lower ones.  In a block, rows of one expert
  // share their weights and columns their rows
  const int used = a.offsets[a.E + 1], groups = (tiles_n + columns - 1) / columns;
  const int k = blockIdx.x >> 3, block = k / (4 * columns) * 8 + (blockIdx.x & 7);
  const int in = k % (4 * columns);
  const int tm = block / groups * 4 + in % 4, tn = block % groups * columns + in / 4;
  if (tm >= used || tn >= tiles_n) return;
  const int e = a.tile_expert[tm], row0 = a.tile_row[tm];
  // up to the expert's next tile or end
  const int tm1 = min(tm + 1, used - 1), e1 = a.tile_expert[tm1], row1 = a.tile_row[tm1];
  const int rows = (tm1 > tm && e1 == e ? row1 : a.offsets[e + 1]) - row0;

  LinearArgs l = {};
  l.out = a.out;
  l.x_stride = a.x_stride;
  l.w_stride = a.K;
  l.out_stride = a.O;
  l.N = GLU ? 2 * a.O : a.O;
  l.K = a.K;
  l.limit = a.limit;
  l.alpha = a.alpha;
  l.offset = a.offset;
  l.cubic = a.cubic;
  const ExpertWork<GLU> work = {a, row0, rows, tn * (GLU ? 128 : 256),
                                (const __bf16*)a.w + (int64_t)e * l.N * a.K};
  constexpr int UNIT = GLU ? LINEAR_GLU : LINEAR_PLAIN;
  if (rows > 224)
    linear_tiles<8, 8, 3, 2, UNIT>(l, work, lds);
  else if (rows > 192)
    linear_tiles<8, 7, 3, 2, UNIT>(l, work, lds);
  else if (rows > 160)
    linear_tiles<8, 6, 3, 2, UNIT>(l, work, lds);
  else if (rows > 128)
    linear_tiles<8, 5, 3, 3, UNIT>(l, work, lds);
  else if (rows > 64)
    linear_tiles<8, 4, 3, 4, UNIT>(l, work, lds);
  else
    linear_tiles<8, 2, 4, 4, UNIT>(l, work, lds);
#endif
}

template <bool GLU>
static void launch(const ExpertsArgs& a, hipStream_t stream) {
  allow_lds<experts_gemm_kernel<GLU>>(LDS_BYTES);
  const int per = GLU ? 128 : 256;
  const int tiles_n = (a.O + per - 1) / per;
  const int groups = (tiles_n + 4) / 5, columns = (tiles_n + groups - 1) / groups;
  const int blocks = (a.tiles + 3) / 4 * ((tiles_n + columns - 1) / columns);
  const int workgroups = (blocks + 7) / 8 * 8 * 4 * columns;
  experts_gemm_kernel<GLU><<<workgroups, 256, LDS_BYTES, stream>>>(a, tiles_n, columns);
}

extern "C" void launch_experts_gemm(bool glu, const ExpertsArgs* a, hipStream_t stream) {
  glu ? launch<true>(*a, stream) : launch<false>(*a, stream);
}
