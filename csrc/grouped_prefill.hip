// Grouped attention of prompt portions over the paged cache on the matrix cores
// (gfx950): windows that keep the first tokens, chunks, capped scores, biases by distance, a
// sink; softmax or sigmoid weights; a gate per head.
//
// A workgroup owns 128 query rows of one head, a wave 32 of them.  Keys and values
// stream through LDS in tiles of 64, double buffered, loaded straight from their pages;
// LDS rows are 16-byte units XOR-swizzled on the source address.  The tiles are those
// of the kept tokens and those of the window; what lies between is never read.
//
//   QK^T (A = keys, B = queries, 32x32x16): a lane owns one query and, per 32
//     keys, the rows (r & 3) + 8 (r >> 2) + 4 (lane >> 5)
//   softmax: 32 registers and one exchange between the lane halves; it starts from
//     the sink (maximum = sink, sum = 1).  Sigmoid weights need neither
//   biases: beyond the last distance with one of its own they are one number a head;
//     only tiles nearer than that look them up
//   PV (A = values^T, B = probabilities): the product's 16 key slots are taken in
//     the order the scores already have, so the probabilities never leave their lane;
//     the value fragments are read transposed (ds_read_b64_tr_b16) in that order
//
// Tiles come heaviest first; the query heads of one key/value head stay on one XCD.
//
// What bounds it (8131 tokens, 32 heads of 128 over 8, no window): products and their LDS
// reads alone take 435 of 613 us (884 TFLOP/s of visible pairs), the softmax and the staging
// the rest, of which two workgroups a CU overlap a part.  720 TFLOP/s before three changes:
// key fragments read three steps ahead of their products (705 -> 645 us), value fragments
// read 16 keys at a time without waiting for the next tile's loads, the first ones before
// the softmax (645 -> 612 us), and scalar page addresses.  No gain: scores of the next tile
// made during the softmax of this one (spills or 720 us), tiles through registers (645 us),
// raised wave priority around the products (626 us), sums of weights as a product (624 us).
// 15 prompts of 700 to 1400 tokens, whose half-empty diagonal tiles weigh more: 264 -> 225 us.
#include "common_t.h"
#include "grouped_attn.h"
#include "launch.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));
typedef float f32x16_v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(1))) const char glob_char;
typedef __attribute__((address_space(4))) const int const_int;

#define KT 64
#define QROWS 128
#define NEG -1e30f
#define LOG2E 1.44269504088896f

template <int N>
struct Int {
  static constexpr int value = N;
};

// the larger of a lane's value and the one of lane ^ 32
static DEV float other_half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}

// FORM: 0 softmax, 1 softmax of capped scores, 2 sigmoid.  PAGED: pages of 16 2^n keys
template <int DN, int VN, int FORM, bool PAGED>
__global__ __launch_bounds__(256, DN + VN <= 4 ? 2 : 1) void grouped_prefill_kernel(
    const GroupedArgs a) {
  constexpr bool CAP = FORM == 1, SIG = FORM == 2;
  constexpr int D = 64 * DN, V = 64 * VN;
  constexpr int KU = D / 8, VU = V / 8;       // units per LDS row
  constexpr int STEPS = D / 16, VT = V / 32;
  constexpr int K_BYTES = KT * D * 2, V_BYTES = KT * V * 2;
  extern __shared__ char lds[];
  int* const slots = (int*)(lds + 2 * (K_BYTES + V_BYTES));  // [2][KT]

  // 8 XCDs take consecutive workgroups in turn: give each its own run of heads
  int head, tile;
  {
    const int id = blockIdx.x;
    if (a.H % 8 == 0) {
      const int per = a.H / 8, slot = id >> 3;
      head = (id & 7) * per + slot % per;
      tile = slot / per;
    } else {
      head = id % a.H;
      tile = id / a.H;
    }
    tile = a.n_tiles - 1 - tile;
  }
  const int kvh = head / (a.H / a.G);
  const int seq = a.tile_seq[tile], q0 = a.tile_q0[tile];
  const int ctx = a.ctx_lens[seq];
  const int rows = min(QROWS, a.seq_lens[seq] - ctx - q0);
  const int64_t row0 = a.row_starts[seq] + q0;
  const int* table = a.tables + (int64_t)seq * a.max_blocks;

  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, half = lane >> 5;
  const int r = wid * 32 + c;
  const bool live = r < rows;
  const int qpos = live ? ctx + q0 + r : -1;

  // key tiles: those with kept tokens, then those some row's window reaches
  const int k_end = ctx + q0 + rows;
  const int kept = (min(a.keep, k_end) + KT - 1) / KT;
  const int first = max(kept, first_key(a, ctx + q0) / KT);
  const int n_tiles = kept + max(0, (k_end + KT - 1) / KT - first);
  auto key_of = [&](int t) { return (t < kept ? t : first + t - kept) * KT; };
  // Keys and values come in 16-byte units, a lane one of them: unit (lane % U) of key
  // (i * 4 + wid) * 64 / U + lane / U of the tile, U units a row.  Keys past the end are the
  // last one again.  With pages of whole groups of 16 keys a group's place is scalar, and a
  // lane's offset in it does not change but at the end; other pages go through a list in LDS.
  const uint32_t k_row = (uint32_t)a.G * D * 2, v_row = (uint32_t)a.G * V * 2;  // bytes
  const char* kp = (const char*)a.k_cache + (int64_t)kvh * D * 2;
  const char* vp = (const char*)a.v_cache + (int64_t)kvh * V * 2;
  const int shift = __builtin_ctz(a.kv_block);
  const const_int* pages = (const const_int*)table;
  struct Groups { int slot[KT / 16]; };  // first slots of a tile's groups of 16 keys
  auto find_groups = [&](int t) {
    Groups s;
#pragma unroll
    for (int i = 0; i < KT / 16; ++i) {
      const int k = min(key_of(t) + i * 16, (k_end - 1) & ~15);
      s.slot[i] = PAGED ? (pages[k >> shift] << shift) + (k & (a.kv_block - 1)) : 0;
    }
    return s;
  };
  auto lane_key = [&](int t) { return min(key_of(t) + lane, k_end - 1); };
  auto find_page = [&](int t) { return table[lane_key(t) / a.kv_block]; };
  auto put_slot = [&](int t, int page) {
    slots[(t & 1) * KT + lane] = page * a.kv_block + lane_key(t) % a.kv_block;
  };

  auto stage = [&](int t, const Groups& at, char* dst, const char* src, uint32_t row, auto units) {
    constexpr int U = decltype(units)::value, KEYS = 64 / U;  // keys of a wave's load
    const int in_group = (wid * KEYS & 15) + lane / U;
    const int sw = in_group & 7;
    const uint32_t unit = ((lane % U) ^ (((sw & 3) << 1) | (sw >> 2))) * 16;
    if constexpr (PAGED) {
      constexpr int STEP = 4 * KEYS;  // keys from one i to the next: 8, 16 or 32
      const int key0 = key_of(t);
      uint32_t offs[U / 4];
#pragma unroll
      for (int i = 0; i < U / 4; ++i)
        offs[i] = (in_group + (STEP == 8 ? (i & 1) * 8 : 0)) * row + unit;
      if (key0 + KT > k_end) {
#pragma unroll
        for (int i = 0; i < U / 4; ++i) {
          const int g = STEP == 32 ? i * 2 + (wid >> 1) : i * STEP / 16;
          const int more = STEP == 8 ? (i & 1) * 8 : 0;
          const int first = min(key0 + g * 16, (k_end - 1) & ~15);
          offs[i] = min(in_group + more, k_end - 1 - first) * row + unit;
          asm volatile("" : "+v"(offs[i]));  // a branch, not selects in every tile
        }
      }
#pragma unroll
      for (int i = 0; i < U / 4; ++i) {
        const int slot = STEP == 32 ? (wid >> 1 ? at.slot[i * 2 % 4 + 1] : at.slot[i * 2 % 4])
                                    : at.slot[i * STEP / 16 % 4];
        __builtin_amdgcn_global_load_lds(
            (glob_char*)(src + (uint64_t)(uint32_t)slot * row + offs[i]),
            (lds_char*)(dst + (i * 4 + wid) * 1024), 16, 0, 0);
      }
    } else {
      const int* sl = slots + (t & 1) * KT + wid * KEYS + lane / U;
      uint32_t slot[U / 4];
#pragma unroll
      for (int i = 0; i < U / 4; ++i) slot[i] = sl[i * 4 * KEYS];
#pragma unroll
      for (int i = 0; i < U / 4; ++i)
        __builtin_amdgcn_global_load_lds(
            (glob_char*)(src + unit + (uint64_t)slot[i] * row),
            (lds_char*)(dst + (i * 4 + wid) * 1024), 16, 0, 0);
    }
  };
  auto stage_k = [&](int t, const Groups& at) {
    stage(t, at, lds + (t & 1) * K_BYTES, kp, k_row, Int<KU>());
  };
  auto stage_v = [&](int t, const Groups& at) {
    stage(t, at, lds + 2 * K_BYTES + (t & 1) * V_BYTES, vp, v_row, Int<VU>());
  };
  Groups at = find_groups(0);
  if (!PAGED) {
    if (wid < 2 && wid < n_tiles) put_slot(wid, find_page(wid));
    __syncthreads();
  }
  stage_k(0, at);
  stage_v(0, at);
  at = find_groups(1);

  // query fragments: 8 consecutive dims of row c per step
  bf16x8_v qf[STEPS];
  {
    const int64_t n = row0 + (live ? r : 0);
    const bf16_t* qr = (const bf16_t*)a.q + n * a.q_stride + (int64_t)head * D + half * 8;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) qf[s] = *(const bf16x8_v*)(qr + s * 16);
    if (!CAP && a.scale < 0.f)
#pragma unroll
      for (int s = 0; s < STEPS; ++s) qf[s] = -qf[s];
  }

  // scores in the exp2 domain: a positive factor, or c1 - 2 c1 / (exp2(c3 s) + 1)
  const float c1 = a.cap * LOG2E;
  const float mul = CAP ? 2.f * LOG2E * a.scale / a.cap : fmaxf(fabsf(a.scale * LOG2E), 1e-30f);
  float m_run = a.sink ? a.sink[head] * LOG2E : NEG;
  float l_run = a.sink && half == 0 ? 1.f : 0.f;
  const float* bias = a.bias ? a.bias + (int64_t)head * a.n_bias : nullptr;
  const int far = a.n_bias - 1;
  const float b_far = bias ? bias[far] * LOG2E : 0.f;
  f32x16_v o[VT] = {};
  const int w_lo = ctx + q0 + wid * 32;                    // wave's positions
  const int w_hi = min(w_lo + 31, k_end - 1);
  const int lo = live ? first_key(a, qpos) : 0;
  const int lo_lo = first_key(a, w_lo), lo_hi = first_key(a, max(w_lo, w_hi));
  const int sw_k = ((c & 3) << 1) | ((c >> 2) & 1);
  const int i16 = lane & 15, g = lane >> 4;
  // a tile that one of this wave's rows sees
  auto seen = [&](int t) {
    const int key0 = key_of(t);
    return t < n_tiles && wid * 32 < rows && key0 <= w_hi &&
           (key0 + KT - 1 >= lo_lo || key0 < a.keep);
  };

  struct Scores { f32x16_v b[2]; };
  auto products = [&](int t, Scores& s) {
    const char* kt = lds + (t & 1) * K_BYTES;
    s = Scores{};
#pragma unroll
    for (int st = 0; st < STEPS; ++st) {
      const int off = ((st * 2 + half) ^ sw_k) << 4;
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const bf16x8_v kf = *(const bf16x8_v*)(kt + (b * 32 + c) * (D * 2) + off);
        s.b[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[st], s.b[b], 0, 0, 0);
      }
    }
    // fragments three steps ahead of their products
    constexpr int AHEAD = STEPS < 3 ? STEPS : 3;
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);  // LDS reads
#pragma unroll
    for (int i = 0; i < STEPS - AHEAD; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);  // products
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x8, 2 * AHEAD, 0);
  };
  // scores of tile t to weights
  auto weights = [&](int t, Scores& s) {
    const int key0 = key_of(t);
    const bool edge = key0 + KT - 1 > w_lo || key0 < lo_hi;
    float add = 0.f, by = 1.f;  // what is left to do: by * score + add
    if (CAP || SIG || bias) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float v = s.b[b][e] * mul;
          if (CAP) v = c1 - 2.f * c1 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v) + 1.f);
          s.b[b][e] = v + b_far;
        }
      if (bias && w_lo - (key0 + KT - 1) < far) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int key = key0 + b * 32 + (e & 3) + 8 * (e >> 2) + 4 * half;
            s.b[b][e] += bias[min(max(qpos - key, 0), far)] * LOG2E - b_far;
          }
      }
    } else {
      by = mul;
    }
    if (edge) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = key0 + b * 32 + (e & 3) + 8 * (e >> 2) + 4 * half;
          s.b[b][e] = (key > qpos) | ((key < lo) & (key >= a.keep)) ? -INFINITY : s.b[b][e];
        }
    }
    if constexpr (SIG) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          s.b[b][e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-s.b[b][e]));
    } else {
      float mt = NEG;
#pragma unroll
      for (int e = 0; e < 16; ++e) mt = fmaxf(fmaxf(mt, s.b[0][e]), s.b[1][e]);
      mt = other_half_max(mt) * by;
      if (__any(mt > m_run)) {
        const float m_new = fmaxf(m_run, mt);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int n = 0; n < VT; ++n) o[n] *= alpha;
      }
      add = -m_run;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          s.b[b][e] = __builtin_amdgcn_exp2f(fmaf(s.b[b][e], by, add));
    }
  };
  // Value fragments of 16 keys.  The builtin for transposed reads would wait for every load
  // in flight, the next tile's too; these wait for themselves.
  struct Values { bf16x4_v lo[VT], hi[VT]; };
  const int sw_v = ((i16 >> 2) << 1) | (g >> 1), unit_v = (g & 1) * 2 + ((i16 & 3) >> 1);
  int at_v[VT];
#pragma unroll
  for (int n = 0; n < VT; ++n)
    at_v[n] = (int)(intptr_t)(lds_char*)lds + 2 * K_BYTES + (4 * (g >> 1) + (i16 >> 2)) * (V * 2) +
              (i16 & 1) * 8 + (((n * 4 + unit_v) ^ sw_v) << 4);
  auto read_values = [&](int t, int ks, Values& v) {
    const int base = (t & 1) * V_BYTES + ks * 16 * (V * 2);
#pragma unroll
    for (int n = 0; n < VT; n += 2) {
      if (VT >= 4 && n % 4) continue;
      const int p0 = at_v[n] + base, p1 = at_v[n + 1] + base;
      if constexpr (VT >= 4) {
        const int p2 = at_v[n + 2] + base, p3 = at_v[n + 3] + base;
        asm volatile(
            "ds_read_b64_tr_b16 %0, %8\n\t"
            "ds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
            "ds_read_b64_tr_b16 %2, %9\n\t"
            "ds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
            "ds_read_b64_tr_b16 %4, %10\n\t"
            "ds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
            "ds_read_b64_tr_b16 %6, %11\n\t"
            "ds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v.lo[n]), "=&v"(v.hi[n]), "=&v"(v.lo[n + 1]), "=&v"(v.hi[n + 1]),
              "=&v"(v.lo[n + 2]), "=&v"(v.hi[n + 2]), "=&v"(v.lo[n + 3]), "=&v"(v.hi[n + 3])
            : "v"(p0), "v"(p1), "v"(p2), "v"(p3), "n"(8 * V * 2)
            : "memory");
      } else {
        asm volatile(
            "ds_read_b64_tr_b16 %0, %4\n\t"
            "ds_read_b64_tr_b16 %1, %4 offset:%6\n\t"
            "ds_read_b64_tr_b16 %2, %5\n\t"
            "ds_read_b64_tr_b16 %3, %5 offset:%6\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v.lo[n]), "=&v"(v.hi[n]), "=&v"(v.lo[n + 1]), "=&v"(v.hi[n + 1])
            : "v"(p0), "v"(p1), "n"(8 * V * 2)
            : "memory");
      }
    }
  };
  // The denominator adds up the weights as the product takes them, rounded: what a weight is off
  // by then cancels in part.  With unrounded ones the error against 64 bits was larger than that
  // of tiles of 32 keys, where more of a row's first weights are 1 and exact: rows of 1 to 900
  // keys 1.993e-3, here 1.978e-3, tiles of 32 1.982e-3.
  auto add_values = [&](int ks, const Scores& s, const Values& v, float& sum) {
    bf16x8_v pf;
#pragma unroll
    for (int e = 0; e < 8; ++e) pf[e] = (__bf16)s.b[ks >> 1][(ks & 1) * 8 + e];
    if constexpr (!SIG) {
      const bf16x2_v one = {(__bf16)1.f, (__bf16)1.f};
#pragma unroll
      for (int e = 0; e < 8; e += 2)
        sum = __builtin_amdgcn_fdot2_f32_bf16(bf16x2_v{pf[e], pf[e + 1]}, one, sum, false);
    }
#pragma unroll
    for (int n = 0; n < VT; ++n) {
      const bf16x8_v vf = __builtin_shufflevector(v.lo[n], v.hi[n], 0, 1, 2, 3, 4, 5, 6, 7);
      o[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[n], 0, 0, 0);
    }
  };

  for (int t = 0; t < n_tiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // tile t landed for every wave; tile t - 1 is fully read
    int page = 0;
    const bool look = !PAGED && wid == 0 && t + 2 < n_tiles;
    if (look) page = find_page(t + 2);
    if (t + 1 < n_tiles) {
      stage_k(t + 1, at);
      stage_v(t + 1, at);
    }
    at = find_groups(t + 2);
    if (seen(t)) {
      Scores s;
      Values v;
      products(t, s);
      read_values(t, 0, v);
      weights(t, s);
      float sum = 0.f;
#pragma unroll
      for (int ks = 0; ks < KT / 16; ++ks) {
        if (ks) read_values(t, ks, v);
        add_values(ks, s, v, sum);
      }
      l_run += sum;
    }
    // their place held tile t's, which were read an iteration ago
    if (look) put_slot(t + 2, page);
  }

  l_run += __shfl_xor(l_run, 32, 64);
  if (!live) return;
  float inv = SIG ? 1.f : l_run > 0.f ? 1.f / l_run : 0.f;
  if (a.gate) inv *= sigmoid_f(bf2f(((const bf16_t*)a.gate)[(row0 + r) * a.gate_stride + head]));
  bf16_t* dst = (bf16_t*)a.out + (row0 + r) * a.out_stride + (int64_t)head * V + 4 * half;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v[4] = {o[t][4 * e] * inv, o[t][4 * e + 1] * inv, o[t][4 * e + 2] * inv,
                          o[t][4 * e + 3] * inv};
      store_f<4>(dst + t * 32 + e * 8, v);
    }
}

template <int DN, int VN, int FORM, bool PAGED>
static void launch_paged(const GroupedArgs& a, hipStream_t stream) {
  constexpr int bytes = 2 * KT * (64 * DN + 64 * VN) * 2 + 2 * KT * 4;
  static_assert(bytes <= 160 * 1024, "LDS");
  allow_lds<grouped_prefill_kernel<DN, VN, FORM, PAGED>>(bytes);
  grouped_prefill_kernel<DN, VN, FORM, PAGED><<<a.n_tiles * a.H, 256, bytes, stream>>>(a);
}

template <int DN, int VN, int FORM>
static void launch(const GroupedArgs& a, hipStream_t stream) {
  const bool paged = a.kv_block >= 16 && (a.kv_block & (a.kv_block - 1)) == 0;
  (paged ? launch_paged<DN, VN, FORM, true> : launch_paged<DN, VN, FORM, false>)(a, stream);
}

template <int DN, int VN>
static bool launch_form(const GroupedArgs& a, hipStream_t stream) {
  if (a.sigmoid && a.cap > 0.f) return false;
  (a.sigmoid       ? launch<DN, VN, 2>
   : a.cap > 0.f   ? launch<DN, VN, 1>
                   : launch<DN, VN, 0>)(a, stream);
  return true;
}

template <int DN>
static bool launch_v(const GroupedArgs& a, int v, hipStream_t stream) {
  switch (v) {
    case 64: return launch_form<DN, 1>(a, stream);
    case 128: return launch_form<DN, 2>(a, stream);
    case 256: return launch_form<DN, 4>(a, stream);
    default: return false;
  }
}

extern "C" bool launch_grouped_prefill(const GroupedArgs* a, int d, int v,
                                       hipStream_t stream) {
  switch (d) {
    case 64: return launch_v<1>(*a, v, stream);
    case 128: return launch_v<2>(*a, v, stream);
    case 256: return launch_v<4>(*a, v, stream);
    default: return false;
  }
}
