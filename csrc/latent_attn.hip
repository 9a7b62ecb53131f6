// Attention of absorbed queries over cached latent rows (gfx950).
//
// A cached row [latent: rank | rotated: 64] is the key of every head, and its
// latent part is the value of every head: one row serves all heads' products
// twice.  Queries are flattened (token, head) rows; a workgroup owns 16*MG of
// them, which for decode are the heads of one sequence.
//
//   tile = 64 keys (32) staged once in LDS by direct global->LDS loads (row-major,
//     16-byte units XOR-swizzled on the source address), double buffered
//   QK^T: wave w takes keys 16w..16w+15, all query rows (A = keys, B = queries,
//     so a lane owns one query row and 4 of its keys)
//   softmax: row maxima cross waves through LDS, probabilities go to LDS as bf16
//   PV: wave w takes latent columns [w*rank/4, ...) for all 64 keys; the value
//     fragments are the same LDS tile read transposed (ds_read_b64_tr_b16)
//
// So each wave reads half of the tile once per product, whatever MG is, and the
// accumulator of a wave is rank/4 columns only.  The swizzle moves 4 consecutive
// keys by 2 units each, which keeps both the row reads (16 keys, one unit) and
// the transposed reads (4 keys, two units) off each other's banks.
//
// Decode of up to 16 heads reads a row once, past the caches: 40 x 200 to 6000 keys 33.1 to 32.5 us.
// Keys past a sequence's end are clamped to its last key and masked; split-K
// partials are merged by split_combine_kernel.  The grid depends on host
// values only (capture-safe); lengths are read on the device.
#include <type_traits>

#include "common_t.h"
#include "latent_attn.h"
#include "launch.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_v __attribute__((ext_vector_type(4)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) bf16x4_v lds_bf16x4;
typedef __attribute__((address_space(1))) const char glob_char;

#define ROT 64         // padded rotated dims
#define NEG -1e30f

// one query tile's place
struct Tile {
  int seq, r0, count, ctx, S, token0;
};

static DEV Tile find_tile(const LatentArgs& a, int rows_per_tile) {
  Tile t;
  if (a.tile_seq) {
    t.seq = a.tile_seq[blockIdx.x];
    t.r0 = a.tile_r0[blockIdx.x];
    t.S = a.seq_lens[t.seq];
    t.ctx = a.ctx_lens[t.seq];
    t.token0 = a.row_starts[t.seq];
  } else {
    const int per_seq = (a.H + rows_per_tile - 1) / rows_per_tile;
    t.seq = blockIdx.x / per_seq;
    t.r0 = (blockIdx.x % per_seq) * rows_per_tile;
    t.S = a.seq_lens[t.seq];
    t.ctx = t.S - 1;
    t.token0 = t.seq;
  }
  t.count = min(rows_per_tile, (t.S - t.ctx) * a.H - t.r0);
  return t;
}

// Sum (or maximum) over the lanes up to this one
template <bool MAX>
static DEV int scan_lanes(int v) {
  auto join = [&](int other) { v = MAX ? max(v, other) : v + other; };
  join(__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));  // row_shr
  join(__builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  join(__builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  join(__builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  join(__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  join(__builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return v;
}

// A decode step's part of a sequence: tiles [index each, (index + 1) each) of its ``parts``
struct Part {
  int seq, len, index, each, parts;
};

// Parts of one size for all sequences, so that long ones have more of them and none is the launch's end alone:
// the size with which the workgroups, n_split a sequence, are enough (each sequence has at most one part
// that is not whole), but none smaller than 128 keys if n_split parts of the longest are not.
// Every workgroup begins with this, so that its length counts (quotient()).
template <int KT>
static DEV Part find_part(const LatentArgs& a, int unit) {
  const int lane = threadIdx.x & 63, per = (a.seqs + 63) / 64;  // sequences of a lane, at most 4
  int len[4] = {}, tiles[4] = {}, sum = 0, most = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= per) break;
    const int s = lane * per + i;
    len[i] = s < a.seqs ? a.seq_lens[s] : 0;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= per) break;
    tiles[i] = (min(len[i], a.window) + KT - 1) / KT;
    sum += tiles[i];
    most = max(most, tiles[i]);
  }
  const int total = __builtin_amdgcn_readlane(scan_lanes<false>(sum), 63);
  const int longest = __builtin_amdgcn_readlane(scan_lanes<true>(most), 63);
  auto parts_of = [](int n, int by) { return quotient(n + by - 1, by); };
  const int even = parts_of(longest, a.n_split);
  const int enough = parts_of(total, (a.n_split - 1) * a.seqs);
  const int each = max(max(min(enough, even), parts_of(longest, a.cap)), max(min(128 / KT, even), 1));
  int parts[4] = {}, mine = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= per) break;
    parts[i] = lane * per + i < a.seqs ? max(1, parts_of(tiles[i], each)) : 0;
    mine += parts[i];
  }
  int before = scan_lanes<false>(mine) - mine;
  const unsigned long long here = __ballot(unit >= before && unit < before + mine);
  if (!here) return {-1, 0, 0, 0, 0};
  int found = 0, index = 0, count = 0, length = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= per) break;
    if (unit >= before && unit < before + parts[i]) {
      found = lane * per + i;
      length = len[i];
      index = unit - before;
      count = parts[i];
    }
    before += parts[i];
  }
  const int from = __builtin_ctzll(here);
  return {__builtin_amdgcn_readlane(found, from), __builtin_amdgcn_readlane(length, from),
          __builtin_amdgcn_readlane(index, from), each, __builtin_amdgcn_readlane(count, from)};
}

// KT: keys of a tile, 16 a wave for the scores.  LENGTHS: a decode step's parts by the sequences' lengths (a.cap >
// a.n_split).  16 heads of rank 512, this kernel alone, us by n_split parts a sequence and by lengths: 40 x 200 to 6000
// keys 43.9 and 33.7, alike 130 x 1000 35.5 and 36.9, 250 x 1000 55.0 and 56.4, of which find_part() is the
// difference; with general divisions in it and for the rows, and with empty parts written first, 34.5, 37.4 and 56.8.
template <int NR, int MG, int KT, bool LENGTHS>
__global__ __launch_bounds__(256, KT == 32 ? 2 : 1) void latent_attn_kernel(const LatentArgs a) {
  constexpr int RANK = 64 * NR;
  constexpr int PPAD = KT + 8;             // probability row in LDS, bf16 elements
  constexpr int ROW = RANK + ROT;
  constexpr int UPR = ROW / 8;             // 16-byte units per row
  constexpr int STEPS = ROW / 32;          // MFMA k-steps of QK^T
  constexpr int TILE_BYTES = KT * ROW * 2;
  constexpr int M = 16 * MG;
  extern __shared__ char lds[];
  bf16_t* const prob = (bf16_t*)(lds + 2 * TILE_BYTES);          // [M][PPAD]
  float* const red = (float*)(prob + M * PPAD);                   // [M][4]
  int* const slots = (int*)(red + M * 4);                         // [2][KT]
  int* const pages = slots + 2 * KT;                              // [2][KT]

  Tile tl;
  Part part = {0, 0, (int)blockIdx.y, 0, 0};
  if constexpr (LENGTHS) {
    const int per_seq = (a.H + M - 1) / M, at = blockIdx.x / per_seq;
    part = find_part<KT>(a, part.index * a.seqs + at);
    if (part.seq < 0) return;
    const int r0 = (blockIdx.x - at * per_seq) * M;
    tl = {part.seq, r0, min(M, a.H - r0), part.len - 1, part.len, part.seq};
  } else {
    tl = find_tile(a, M);
  }
  const int split = part.index;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const bf16_t* cache = (const bf16_t*)a.cache;
  const int* table = a.tables + (int64_t)tl.seq * a.max_blocks;

  // keys any row of the tile sees
  auto token_of = [&](int r) { return LENGTHS ? 0 : r / a.H; };  // of the tile's sequence
  const int pos_lo = tl.ctx + token_of(tl.r0);
  const int pos_hi = tl.ctx + token_of(tl.r0 + tl.count - 1);
  const int k_begin = max(0, pos_lo - a.window + 1);
  const int k_end = pos_hi + 1;
  const int n_tiles = (k_end - k_begin + KT - 1) / KT;
  const int per_split = LENGTHS ? part.each : (n_tiles + a.n_split - 1) / a.n_split;
  const int t_begin = min(n_tiles, split * per_split);
  const int t_end = min(n_tiles, t_begin + per_split);

  const int64_t row0 = (int64_t)tl.token0 * a.H + tl.r0;
  // empty splits; those are a row's last ones
  auto no_parts = [&](int from, int to) {
    for (int i = threadIdx.x; i < (to - from) * M; i += 256)
      if (i % M < tl.count) a.part_ml[(int64_t)(from + i / M) * a.rows + row0 + i % M] = float2{NEG, -1.f};
  };
  if (t_begin >= t_end) {
    no_parts(split, LENGTHS ? a.cap : split + 1);
    return;
  }

  // B fragments of the queries: lane's row c, 8 consecutive dims per step
  bf16x8_v qf[MG][STEPS];
  int qpos[MG];
#pragma unroll
  for (int m = 0; m < MG; ++m) {
    const int r = m * 16 + c;
    const bool live = r < tl.count;
    qpos[m] = live ? tl.ctx + token_of(tl.r0 + r) : -1;  // -1 sees no key
    const int64_t row = row0 + (live ? r : 0);
    const int64_t token = LENGTHS ? tl.token0 : row / a.H;
    const bf16_t* qr = (const bf16_t*)a.q + row * RANK + g * 8;
#pragma unroll
    for (int s = 0; s < RANK / 32; ++s) qf[m][s] = *(const bf16x8_v*)(qr + s * 32);
    // the rest is rotated on the way in: 4 pairs a lane and step
    const bf16_t* rr = (const bf16_t*)a.q_rot + token * a.rot_token + (row - token * a.H) * a.rot_head + g * 8;
    const int pairs = a.rot_dim >> 1;
    const float* ct = a.cos_sin + (int64_t)max(qpos[m], 0) * pairs;
    const float* st = ct + a.positions * pairs;
#pragma unroll
    for (int s = 0; s < ROT / 32; ++s) {
      bf16x8_v q8 = *(const bf16x8_v*)(rr + s * 32);
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int i = min(s * 16 + g * 4 + p, pairs - 1);  // padding is zero: any angle
        const float x = (float)q8[2 * p], y = (float)q8[2 * p + 1];
        q8[2 * p] = (__bf16)(x * ct[i] - y * st[i]);
        q8[2 * p + 1] = (__bf16)(y * ct[i] + x * st[i]);
      }
      qf[m][RANK / 32 + s] = q8;
    }
  }

  // Where a CU has two workgroups pages go from the tables to LDS, three tiles ahead, and become slots two
  // tiles ahead: in registers they would be waited for, and with them, as loads come back in order, all of
  // the tile behind them.  A workgroup alone does not gain by it: 129 x 4096 keys of 32 heads 244 us so,
  // 233 by registers and barriers that wait for the tile
  constexpr bool APART = KT == 32;
  auto key_of = [&](int t) { return min(k_begin + t * KT + (int)threadIdx.x, k_end - 1); };
  auto ask_pages = [&](int t) {
    if (threadIdx.x < KT)
      __builtin_amdgcn_global_load_lds((glob_char*)(table + key_of(t) / a.kv_block),
                                       (lds_char*)(pages + (t & 1) * KT), 4, 0, 0);
  };
  auto put_slots = [&](int t, const int* from) {
    if (threadIdx.x < KT)
      slots[(t & 1) * KT + threadIdx.x] = *from * a.kv_block + key_of(t) % a.kv_block;
  };
  // piece = 1 KiB of the tile image; lane-linear in LDS, swizzled at the source
  auto stage = [&](int t) {
    char* dst = lds + (t & 1) * TILE_BYTES;
#pragma unroll
    for (int i = 0; i < TILE_BYTES / 4096; ++i) {
      const int piece = i * 4 + wid;
      const int u = piece * 64 + lane;
      const int key = u / UPR;
      const int sw = ((key & 3) << 1) | ((key >> 2) & 1);
      const int unit = (u - key * UPR) ^ sw;
      const bf16_t* src = cache + (int64_t)slots[(t & 1) * KT + key] * ROW + unit * 8;
      __builtin_amdgcn_global_load_lds((glob_char*)src, (lds_char*)(dst + piece * 1024),
                                       16, 0, MG == 1 ? 2 : 0);
    }
  };

  put_slots(t_begin, table + key_of(t_begin) / a.kv_block);
  put_slots(t_begin + 1, table + key_of(t_begin + 1) / a.kv_block);
  __syncthreads();
  if constexpr (APART) ask_pages(t_begin + 2);
  stage(t_begin);

  f32x4_v o[MG][NR] = {};
  // a sink is the softmax's starting state: its maximum, one term of the sum, no value
  const bool sink = a.sink && split == 0;
  float m_run[MG], l_run[MG];
#pragma unroll
  for (int m = 0; m < MG; ++m) {
    m_run[m] = sink ? a.sink[(tl.r0 + m * 16 + c) % a.H] * 1.44269504088896f : NEG;
    l_run[m] = sink && wid == 0 && g == 0 ? 1.f : 0.f;
  }
  const float scale2 = a.scale * 1.44269504088896f;  // exp2 domain
  const int sw_c = ((c & 3) << 1) | ((c >> 2) & 1);

  // LDS writes of all waves are done, but not the loads of the next tile, which __syncthreads() waits for
  auto meet = [] {
    if constexpr (APART) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    } else {
      __syncthreads();
    }
  };
  for (int t = t_begin; t < t_end; ++t) {
    // tile t landed for every wave; tile t-1 is fully read
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    meet();
    if constexpr (APART)
      if (t + 3 < t_end) ask_pages(t + 3);
    if (t + 1 < t_end) stage(t + 1);
    const char* tile = lds + (t & 1) * TILE_BYTES;

    // scores: lane holds query row c, keys wid*16 + 4g + {0..3}
    f32x4_v s[MG] = {};
    const bool scores = KT == 64 || wid * 16 < KT;
    if (scores) {
      const char* krow = tile + (wid * 16 + c) * (ROW * 2);
#pragma unroll
      for (int st = 0; st < STEPS; ++st) {
        const bf16x8_v kf = *(const bf16x8_v*)(krow + (((st * 4 + g) ^ sw_c) << 4));
#pragma unroll
        for (int m = 0; m < MG; ++m)
          s[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[m][st], s[m], 0, 0, 0);
      }
    }
    const int key0 = k_begin + t * KT + wid * 16 + 4 * g;
#pragma unroll
    for (int m = 0; m < MG; ++m) {
      float mt = NEG;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = key0 + r;
        const bool see = scores && key <= qpos[m] && qpos[m] - key < a.window;
        s[m][r] = see ? s[m][r] * scale2 : -INFINITY;
        mt = fmaxf(mt, s[m][r]);
      }
      mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
      if (g == 0) red[(m * 16 + c) * 4 + wid] = mt;
    }
    meet();
#pragma unroll
    for (int m = 0; m < MG; ++m) {
      const float4 w4 = *(const float4*)(red + (m * 16 + c) * 4);
      const float m_new = fmaxf(m_run[m], fmaxf(fmaxf(w4.x, w4.y), fmaxf(w4.z, w4.w)));
      const float alpha = __builtin_amdgcn_exp2f(m_run[m] - m_new);
      m_run[m] = m_new;
      float p[4], sum = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[r] = __builtin_amdgcn_exp2f(s[m][r] - m_new);
        sum += p[r];
      }
      l_run[m] = l_run[m] * alpha + sum;
      if (scores) store_f<4>(prob + (m * 16 + c) * PPAD + wid * 16 + 4 * g, p);
#pragma unroll
      for (int n = 0; n < NR; ++n) o[m][n] *= alpha;
    }
    if (t + 2 < t_end)  // tile t's slots were consumed by its stage
      put_slots(t + 2, APART ? pages + (t & 1) * KT + threadIdx.x : table + key_of(t + 2) / a.kv_block);
    meet();

    // values: A = latent columns (transposed read), B = probabilities
#pragma unroll
    for (int ks = 0; ks < KT / 32; ++ks) {
      bf16x8_v pf[MG];
#pragma unroll
      for (int m = 0; m < MG; ++m)
        pf[m] = *(const bf16x8_v*)(prob + (m * 16 + c) * PPAD + ks * 32 + g * 8);
      const int key = ks * 32 + g * 8 + (c >> 2);  // and key + 4
      const int sw_lo = (key & 3) << 1;             // (key >> 2) & 1 == 0 here
      const char* v0 = tile + key * (ROW * 2) + (c & 1) * 8;
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        const int unit = (wid * NR + n) * 2 + ((c & 3) >> 1);
        const bf16x4_v lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (lds_bf16x4*)(v0 + ((unit ^ sw_lo) << 4)));
        const bf16x4_v hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (lds_bf16x4*)(v0 + 4 * (ROW * 2) + ((unit ^ (sw_lo | 1)) << 4)));
        const bf16x8_v vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int m = 0; m < MG; ++m)
          o[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[m], o[m][n], 0, 0, 0);
      }
    }
  }

  // row sums over the lane groups and waves
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MG; ++m) {
    float l = l_run[m];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) red[(m * 16 + c) * 4 + wid] = l;
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MG; ++m) {
    const int r = m * 16 + c;
    if (r >= tl.count) continue;
    const float4 w4 = *(const float4*)(red + r * 4);
    const float l = w4.x + w4.y + w4.z + w4.w;
    const int64_t row = row0 + r;
    const int col0 = wid * (16 * NR) + 4 * g;
    if (a.n_split == 1) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      bf16_t* dst = (bf16_t*)a.out + row * RANK + col0;
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        const float v[4] = {o[m][n][0] * inv, o[m][n][1] * inv, o[m][n][2] * inv,
                            o[m][n][3] * inv};
        store_f<4>(dst + n * 16, v);
      }
    } else {
      const int64_t at = (int64_t)split * a.rows + row;
      if (wid == 0 && g == 0) a.part_ml[at] = float2{m_run[m], l};
      float* dst = a.part + at * RANK + col0;
#pragma unroll
      for (int n = 0; n < NR; ++n) *(f32x4_v*)(dst + n * 16) = o[m][n];
    }
  }
  if (LENGTHS && split == 0) no_parts(part.parts, a.cap);  // no load waits for it here
}

// Merge the splits (at most 64) of one row.
__global__ __launch_bounds__(128) void split_combine_kernel(
    const SplitOut dst, const float* __restrict__ part, const float2* __restrict__ part_ml,
    const int rows, const int rank, const int n_split) {
  __shared__ float weight[64];
  const int row = blockIdx.x, lane = threadIdx.x & 63;
  const float2 ml = lane < n_split ? part_ml[(int64_t)lane * rows + row] : float2{NEG, -1.f};
  const int live = __popcll(__ballot(ml.y >= 0.f));
  const float m = wave_max(ml.x);
  const float w = ml.y > 0.f ? __builtin_amdgcn_exp2f(ml.x - m) : 0.f;
  const float l = wave_sum(w * fmaxf(ml.y, 0.f));
  const int token = row / dst.H, head = row % dst.H;
  if (threadIdx.x < 64) weight[lane] = l > 0.f ? w / l : 0.f;
  bf16_t* out = (bf16_t*)dst.out + token * dst.out_stride + (int64_t)head * rank;
  __syncthreads();
  for (int i = threadIdx.x * 4; i < rank; i += 512) {
    float acc[4] = {};
    const float* src = part + (int64_t)row * rank + i;
#pragma unroll 8
    for (int s = 0; s < live; ++s) {
      float v[4];
      load_f<4>(v, src + (int64_t)s * rows * rank);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] += weight[s] * v[k];
    }
    store_f<4>(out + i, acc);
  }
}

// Plain kernel for fp32 models and latents beyond the MFMA sizes: one workgroup
// per query row, its 4 waves stride over the keys, a lane holds every 64th dim.
template <typename T, int NE>
__global__ __launch_bounds__(256) void latent_attn_plain_kernel(
    const LatentArgs a, const int rank, const int row) {
  const Tile tl = find_tile(a, 1);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t qrow = (int64_t)tl.token0 * a.H + tl.r0;
  const int pos = tl.ctx + tl.r0 / a.H;
  const int* table = a.tables + (int64_t)tl.seq * a.max_blocks;
  float q[NE], acc[NE] = {};
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int d = e * 64 + lane;
    q[e] = 0.f;
    if (d < rank) {
      q[e] = to_f(((const T*)a.q)[qrow * rank + d]) * a.scale;
    } else if (d < rank + a.rot_dim) {
      const int i = (d - rank) >> 1;
      const T* pair = (const T*)a.q_rot + qrow / a.H * a.rot_token +
                      qrow % a.H * a.rot_head + 2 * i;
      const int64_t at = (int64_t)pos * (a.rot_dim >> 1) + i;
      const float co = a.cos_sin[at];
      const float si = a.cos_sin[a.positions * (a.rot_dim >> 1) + at];
      const float u = to_f(pair[0]), v = to_f(pair[1]);
      q[e] = (d & 1 ? v * co + u * si : u * co - v * si) * a.scale;
    }
  }
  const bool sink = a.sink && wid == 0;
  float m = sink ? a.sink[qrow % a.H] : NEG, l = sink ? 1.f : 0.f;
  for (int k = max(0, pos - a.window + 1) + wid; k <= pos; k += 4) {
    const int64_t slot = (int64_t)table[k / a.kv_block] * a.kv_block + k % a.kv_block;
    const T* kr = (const T*)a.cache + slot * row;
    float kv[NE], dot = 0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int d = e * 64 + lane;
      kv[e] = d < row ? to_f(kr[d]) : 0.f;
      dot += q[e] * kv[e];
    }
    dot = wave_sum(dot);
    const float mn = fmaxf(m, dot);
    const float alpha = __expf(m - mn), p = __expf(dot - mn);
    m = mn;
    l = l * alpha + p;
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[e] = acc[e] * alpha + p * kv[e];
  }
  __shared__ float part[4][NE * 64];
  __shared__ float2 ml[4];
#pragma unroll
  for (int e = 0; e < NE; ++e) part[wid][e * 64 + lane] = acc[e];
  if (lane == 0) ml[wid] = float2{m, l};
  __syncthreads();
  float mx = NEG, w[4], sum = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) mx = fmaxf(mx, ml[i].x);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    w[i] = __expf(ml[i].x - mx);
    sum += w[i] * ml[i].y;
  }
  for (int d = threadIdx.x; d < rank; d += 256) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) v += w[i] * part[i][d];
    ((T*)a.out)[qrow * rank + d] = from_f<T>(v / sum);
  }
}

template <int NR, int MG, int KT>
static void launch_tiles(const LatentArgs& a, int tiles, hipStream_t stream) {
  constexpr int M = 16 * MG;
  constexpr int bytes = 2 * KT * (64 * NR + ROT) * 2 + M * (KT + 8) * 2 + M * 16 + 4 * KT * 4;
  static_assert(bytes <= 160 * 1024, "LDS");
  auto launch = [&](auto lengths) {
    constexpr bool LENGTHS = decltype(lengths)::value;
    allow_lds<latent_attn_kernel<NR, MG, KT, LENGTHS>>(bytes);
    latent_attn_kernel<NR, MG, KT, LENGTHS><<<dim3(tiles, a.n_split), 256, bytes, stream>>>(a);
  };
  if (a.cap > a.n_split)
    launch(std::true_type());
  else
    launch(std::false_type());
}

// A tile is a chain of reads, products and three barriers, during which a CU with one workgroup waits:
// with tiles of 32 keys of a wide latent it has two, where there are more than CUs.  40 x 200 to 6000 keys
// of 16 heads 72 us by 64 keys, 57 by 32; four tiles in LDS, three of them under way, of one workgroup a
// CU 91.  By 32 keys alone a step over 1 x 5000 1671 us, else 1651, over 8 x 200 to 800 1928 and 1893.
// A few more than CUs wait for the longest of them, which is slower by 32 keys: 257 x 200 to 2000 99 us by
// 64 keys, 114 by 32, 270 of them 122 and 120; of 100 to 500 34.8 and 36.2, 45.3 and 37.1.
#define CUS 256
template <int NR, int MG>
static void launch_mfma(const LatentArgs& a, int tiles, hipStream_t stream) {
  if constexpr (MG == 1 && NR >= 4)
    if (tiles * (int64_t)a.n_split > CUS + CUS / 32) return launch_tiles<NR, MG, 32>(a, tiles, stream);
  launch_tiles<NR, MG, 64>(a, tiles, stream);
}

template <int NR>
static void launch_mg(const LatentArgs& a, int mg, int tiles, hipStream_t stream) {
  if (mg == 1)
    launch_mfma<NR, 1>(a, tiles, stream);
  else if (mg == 2 || NR > 4)  // query fragments of 64 rows x 448+ dims would spill
    launch_mfma<NR, 2>(a, tiles, stream);
  else if constexpr (NR <= 4)
    launch_mfma<NR, 4>(a, tiles, stream);
}

template <typename T>
static bool launch_plain(const LatentArgs& a, int rank, int row, int tiles,
                         hipStream_t stream) {
  const int ne = (row + 63) / 64;
  if (ne > 32) return false;
  auto k = ne <= 2    ? latent_attn_plain_kernel<T, 2>
           : ne <= 4  ? latent_attn_plain_kernel<T, 4>
           : ne <= 9  ? latent_attn_plain_kernel<T, 9>
           : ne <= 16 ? latent_attn_plain_kernel<T, 16>
                      : latent_attn_plain_kernel<T, 32>;
  k<<<tiles, 256, 0, stream>>>(a, rank, row);
  return true;
}

extern "C" {

void launch_split_combine(const SplitOut* out, const float* part, const float2* part_ml,
                          int rows, int width, int n_split, hipStream_t stream) {
  split_combine_kernel<<<rows, 128, 0, stream>>>(*out, part, part_ml, rows, width, n_split);
}

bool launch_latent_attn(bool bf16, bool mfma, const LatentArgs* a, int rank, int row,
                        int mg, int tiles, bool merge, hipStream_t stream) {
  if (!mfma)
    return (bf16 ? launch_plain<bf16_t> : launch_plain<float>)(*a, rank, row, tiles, stream);
  switch (rank) {
    case 64: launch_mg<1>(*a, mg, tiles, stream); break;
    case 128: launch_mg<2>(*a, mg, tiles, stream); break;
    case 256: launch_mg<4>(*a, mg, tiles, stream); break;
    case 384: launch_mg<6>(*a, mg, tiles, stream); break;
    case 512: launch_mg<8>(*a, mg, tiles, stream); break;
    default: return false;
  }
  if (a->n_split > 1 && merge) {
    const SplitOut out = {a->out, (int64_t)a->H * rank, a->H};
    launch_split_combine(&out, a->part, a->part_ml, a->rows, rank, a->cap, stream);
  }
  return true;
}

}  // extern "C"
