// Launch arguments of the mixture-of-experts kernels (experts.hip, experts_gemm.hip).
#pragma once
#include <hip/hip_runtime.h>

// One product of the routed experts.  An entry is a (token, choice) pair, number
// token * top + choice; entries are grouped by expert through perm.
struct ExpertsArgs {
  void* out;            // gate_up: [entries, O] in grouped order; down: [entries, O] by entry
  const void* x;        // gate_up: [tokens, K] rows x_stride apart; down: [entries, K] grouped
  const void* w;        // gate_up: [E, 2 O, K], gate rows then up rows; down: [E, O, K]
  const int* ids;       // [entries] expert
  const int* perm;      // [entries] entry of a grouped row
  const int* offsets;   // [E + 2] first grouped row of an expert; then the tiles in use
  const int* tile_expert;  // [tiles]
  const int* tile_row;     // [tiles] first grouped row of the tile
  int64_t x_stride;
  int entries, E, O, K, top, tiles;
  float limit, alpha, offset, cubic;  // gate_up: the gated unit
};

// Sizes of the two tiled products: inner elements and columns of workgroups of a tile
struct TiledProducts {
  int width, columns1;  // gate and up
  int inner, columns2;  // down
  bool even;            // an expert's tiles have the same height
};

// rows of one tile of the large-batch product, at most TALL_TILE
#define EXPERT_TILE 256
#define TALL_TILE 320

// Rows of an expert's tiles: even ones of 257 to 320 rows if they cover the expert in fewer tiles,
// as a small last tile takes all of the expert's weights once more.
__device__ static inline int tall_tile(int rows) {
  const int tiles = (rows + TALL_TILE - 1) / TALL_TILE;
  const int even = tiles > 0 ? (rows + tiles - 1) / tiles : 0;
  return even > EXPERT_TILE ? even : EXPERT_TILE;
}
