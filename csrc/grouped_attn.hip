// Grouped attention over the paged cache, one token per sequence, and the plain kernel
// for every other case (gfx950).
//
// A query at position p sees the keys p - window + 1 .. p and the first ``keep``
// ones, or of those only the ones of its own chunk; scores may be mixed over the heads (the
// plain kernel; talk_attn.hip has the others), capped, get a bias by distance, and a sink
// may join the denominator.  The sink is the softmax's starting state (maximum = sink, sum = 1, no
// value), so that neither the merge of partial sums nor the output knows about it.
// Sigmoid weights need no such state: their partial results are plain sums.
//
// Decode: the keys stream once, from memory to registers.  A wave takes 32 of them at a time,
// the next 32 in flight meanwhile: keys as the matrix cores want them (16 keys by 8 dims a lane),
// the heads that share them are the columns of one product; values as 8 dims a lane, weighted in
// fp32 by the VALU.  Between the two the weights pass through a few LDS rows of the wave.
// The blocks of 32 that the sequences' queries see are cut into even shares of the workgroups that are resident at
// once, whatever the lengths (Cut, below); a workgroup finds its share from the lengths by itself, and a
// second launch merges sequences of several workgroups.
// Bound by memory: with the merge 5.9 TB/s of keys and values at 64 x 4096, 6.2 at 256 x 1024 tokens, 32
// heads over 8; 61 x 310 to 4000 106.5 -> 101 us by even shares of all keys, 61 x 670 to 7900 201 -> 184, 13 x
// 300 to 3900 of 32 key heads 86 -> 80.6, but one of 4001 13.1 -> 13.4 and 4 x 200 to 4000 18.8 -> 19.1, whose
// workgroups find the same pieces by a longer way.
// Before, with products and sums over dims on the VALU, 4.1 TB/s there and 2.0 to 3.0 where
// lengths differ: 61 x 310 to 4000 tokens 268 -> 122 us, 190 x 700 to 1300 265 -> 159,
// 1 x 4002 203 -> 14; with the values' loads, whole lines each, past the caches 190 x 700 to 1300 148
// -> 139, 61 x 310 to 4000 120 -> 112.5, and 13 x 300 to 3900 of 32 key heads 95 -> 88; with the
// keys' loads likewise, instead of 16 rows of half a line, 137, 109 and 85, 200 x 100 to 1000 of 64
// heads over 8 130 -> 116; 64 x 128 17.1 -> 16.7, 64 x 16 7.3 -> 7.7 (launches and their first loads, not memory).  Without the next block in
// flight the same kernel takes 350 us at 190 x 700 to 1300; at 3 waves a SIMD the registers for
// it are not there.
#include <type_traits>

#include "common_t.h"
#include "grouped_attn.h"

#define NEG -1e30f
#define LOG2E 1.44269504088896f

struct KeyList {  // of one query: position of the i-th visible key
  int keep, lo, n;
  DEV int at(int i) const { return i < keep ? i : lo + i - keep; }
};

static DEV KeyList visible_keys(const GroupedArgs& a, int pos) {
  KeyList k;
  k.lo = first_key(a, pos);
  k.keep = min(a.keep, k.lo);
  k.n = k.keep + pos + 1 - k.lo;
  return k;
}

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(4))) const int const_int;

#define KB 32  // keys of a block: one wave's step

// The blocks that a query at position pos sees: those with kept tokens, then those its window
// or chunk reaches.
struct Blocks {
  int kept, first, n;
  DEV int key(int i) const { return (i < kept ? i : first + i - kept) * KB; }
};

static DEV Blocks visible_blocks(const GroupedArgs& a, int pos) {
  Blocks b;
  b.kept = (min(a.keep, pos + 1) + KB - 1) / KB;
  b.first = max(b.kept, first_key(a, pos) / KB);
  b.n = b.kept + max(0, (pos + KB) / KB - b.first);
  return b;
}

// A sequence's blocks, one if it has none, or pieces (``n``), and those of the sequences ahead of it
struct Stretch {
  int seq, len, n, before;
};

// sum of the lanes up to this one (row shifts and broadcasts of rows' last lanes)
static DEV int wave_scan(int v) {
#define SCAN(ctrl, rows) v += __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xf, false)
  SCAN(0x111, 0xf); SCAN(0x112, 0xf); SCAN(0x114, 0xf); SCAN(0x118, 0xf);
  SCAN(0x142, 0xa); SCAN(0x143, 0xc);
#undef SCAN
  return v;
}

// a value and the one of lane ^ 16 or lane ^ 32
template <int LANES>
static DEV float2 with_lane(float v) {
  const int i = __float_as_int(v);
  const auto r = LANES == 32 ? __builtin_amdgcn_permlane32_swap(i, i, false, false)
                             : __builtin_amdgcn_permlane16_swap(i, i, false, false);
  return float2{__int_as_float(r[0]), __int_as_float(r[1])};
}
template <int LANES>
static DEV float sum_with(float v) {
  if constexpr (LANES < 16) return v + __shfl_xor(v, LANES, 64);
  const float2 r = with_lane<LANES < 16 ? 16 : LANES>(v);
  return r.x + r.y;
}
template <int LANES>
static DEV float max_with(float v) {
  const float2 r = with_lane<LANES>(v);
  return fmaxf(r.x, r.y);
}

// How a step's blocks are cut for the a.pieces workgroups of a key head.
//
// Into ranges of all sequences' blocks, one after the other, whatever the sequences: a workgroup's
// parts of sequences follow each other, and all workgroups, which are resident at once, end at about the
// same time.  Of many blocks a workgroup has two ranges half as long, of two key heads, as rows
// of some heads come more slowly than others (XCDs and channels share unevenly: one head each, 64 x 2048
// keys end after 68 to 93 us, two 64 to 87).  61 x 310 to 4000 keys of 8 heads, the kernel alone: pieces of
// sequences, up to 1112 workgroups in turn, 105 us, ranges 98, of two heads 93 (on a faster card 92 and 85).
//
// Or few blocks into pieces of one sequence each, where that leaves no workgroup with much more than its share:
// parts have starts and ends, 4 x 300 keys 16.0 us by ranges and 11.8 by pieces, 64 x 512 35.4 and 32.
//
// Without a.ranges always pieces: of one size where they are all resident at once, or sequences are no longer than
// that (16 query heads of 2 key heads, 61 x 310 to 4000 keys, 40.3 us, else 48.4).  Else for about two rounds, with a
// last piece of under a quarter shared by the sequence's others from a.shared_from blocks on (of 12 blocks 20 x 130
// to 3900 keys shared 53.7 us and 52.0 not, of 256 dims, where a CU has one workgroup, 24 x 510 to 2400 104 and 114).
// Without that sharing 64 query heads of 8 key heads, 30 x 300 to 4000 keys, 76.6 us instead of 73.2, 100 x 700 to
// 1300 107.2 and 104.5; 128 query heads, 20 x 130 to 3900 80.0 and 75.2.  The kernel with several parts is 0.5 to
// 1 us slower for one, so that few sequences go without (RANGES_FROM), and for 8 query heads a workgroup it has not
// the registers.
struct Cut {
  bool aligned;  // pieces of sequences
  int count;     // ranges of a workgroup
  int each;      // blocks of a range, at most of a piece of the sequence
};

// Finds the cut and the sequence ``want``, or the one with the first block of workgroup ``item`` of a
// key head (seq < 0: it has none).  A wave's lanes read the lengths, 64 at a time.  Every workgroup begins
// with this and then waits for its first keys, so that its length counts: with general divisions and a
// length read twice 64 x 128 keys took 16.6 us instead of 15.5.
static DEV Stretch find_range(const GroupedArgs& a, int want, int item, Cut& cut) {
  const int lane = threadIdx.x & 63;
  auto len_of = [&](int seq) { return seq < a.seqs ? a.seq_lens[seq] : 0; };
  auto blocks_of = [&](int seq, int len) {  // an empty sequence has a turn, too
    return seq < a.seqs ? max(1, visible_blocks(a, len - 1).n) : 0;
  };
  const int len0 = len_of(lane), mine0 = blocks_of(lane, len0);
  int total = mine0, longest = mine0;
  for (int s = 64; s < a.seqs; s += 64) {
    const int n = blocks_of(s + lane, len_of(s + lane));
    total += n;
    longest = max(longest, n);
  }
  total = __builtin_amdgcn_readlane(wave_scan(total), 63);
  const int spare = a.pieces - a.seqs;
  const bool one_round = a.seqs <= 64 || spare >= 0;  // that they may fit in it
  const int share = a.ranges || one_round ? quotient(total + a.pieces - 1, a.pieces) : 0;
  int few = 0, few_upto = 0;
  int two_rounds = 0;  // blocks of a piece of two rounds
  bool known = false;
  cut.aligned = false;
  cut.count = 1;
  cut.each = max(4, share);
  if (!a.ranges || (share <= 32 && spare >= 0)) {
    const int even = share + 3 & ~3, most = share + share / 4 + 4;
    cut.aligned = true;
    if (a.seqs <= 64) {
      few = quotient(mine0 + even - 1, even);
      few_upto = wave_scan(few);
      known = __builtin_amdgcn_readlane(few_upto, 63) <= a.pieces;
    }
    if (known) {
      cut.each = even;
    } else if (spare >= 0 && !__any(longest > most)) {  // whole sequences
      cut.each = most;
    } else if (!a.ranges) {  // at most 2 a.pieces and one for every sequence; long parts are too uneven
      const int half = max(1, quotient(total + 4 * a.pieces - 1, 4 * a.pieces));
      two_rounds = 4 * (__any(longest > 4 * half) ? max(min(half, 3), (half + 1) / 2) : half);
    } else {
      const int each = spare > 0 ? quotient(total + spare - 1, spare) : most + 1;
      cut.aligned = each <= most;
      if (cut.aligned) cut.each = max(4, each);
    }
  } else if (share > 32 && !(a.G * ((a.group + a.gm - 1) / a.gm) & 1)) {
    cut.count = 2;
    cut.each = (share + 1) / 2;
  }
  const int first = cut.aligned ? item : item * cut.count * cut.each;
  const int spared = two_rounds - (two_rounds < a.shared_from ? 0 : two_rounds / 4) - 1;
  Stretch x = {-1, 0, 0, 0};
  int before = 0;
  for (int s = 0; s < a.seqs; s += 64) {
    const int len = s ? len_of(s + lane) : len0, n = s ? blocks_of(s + lane, len) : mine0;
    int mine = n, each = cut.each;
    if (known) {
      mine = few;
    } else if (two_rounds) {
      mine = max(1, quotient(n + spared, each = two_rounds));
      if (mine * each < n) {
        each = 4 * quotient(n + 4 * mine - 1, 4 * mine);
        mine = quotient(n + each - 1, each);
      }
      if (s + lane >= a.seqs) mine = 0;
    } else if (cut.aligned) {
      mine = quotient(n + each - 1, each);
    }
    const int upto = known ? few_upto : before + wave_scan(mine);  // blocks or pieces up to this lane's
    const uint64_t hit = __ballot(want >= 0 ? s + lane == want : first < upto);
    if (hit) {
      const int at = __builtin_ctzll(hit);
      x.seq = s + at;
      x.len = __builtin_amdgcn_readlane(len, at);
      x.n = __builtin_amdgcn_readlane(mine, at);
      cut.each = __builtin_amdgcn_readlane(each, at);
      x.before = __builtin_amdgcn_readlane(upto, at) - x.n;
      break;
    }
    before = __builtin_amdgcn_readlane(upto, 63);
  }
  return x;
}

// PAGED: pages of 16 2^n keys, so that a group of 16 keys has one, scalar, place.  CUT: the blocks are
// cut (a.pieces > 0), else a workgroup has a sequence.  RANGES: as a.ranges
template <int DN, int VN, int GM, bool SIG, bool PAGED, bool CUT, bool RANGES>
__global__ __launch_bounds__(256, DN + VN <= 4 ? 2 : 1) void grouped_decode_kernel(const GroupedArgs a) {
  constexpr int D = 64 * DN, V = 64 * VN, STEPS = D / 32;
  constexpr int LPK = V / 8, KPL = 64 / LPK, NV = KB / KPL;  // lanes a key, keys a load, loads
  constexpr bool AHEAD = D + V <= 256;  // the next block's loads fit beside this one's
  __shared__ float weight[4][KB][GM], rescale[4][GM];
  __shared__ float lds_acc[4][GM][V];
  __shared__ float2 lds_ml[4][GM];
  __shared__ int slots[PAGED ? 1 : 4][KB];
  const int group = a.group, per = (group + GM - 1) / GM;  // workgroups per kv head
  // Whole sequences of up to 8 workgroups stay on one XCD, whose L2 then sees whole rows of the
  // cache: 190 x 700 to 1300 keys of 8 heads 152 to 148 us, 230 x 500 to 3500 367 to 352, but of 32
  // heads 60 x 100 to 800 89 to 102, and ranges 3% slower
  const int workgroups = per * a.G;  // of the same keys
  const int even = !CUT && workgroups <= 8 ? a.seqs & ~7 : 0;
  const bool near_by = (int)blockIdx.x < even * workgroups;
  const int nth_wg = near_by ? blockIdx.x >> 3 : blockIdx.x - even * workgroups;
  const int nth_item = nth_wg / workgroups, first_at = nth_wg - nth_item * workgroups;
  const int item = near_by ? nth_item * 8 + (blockIdx.x & 7) : even + nth_item;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, j = lane >> 4;           // product: column (head), rows 4 j ..
  const int kl = lane / LPK, el = lane % LPK;       // values: key of a load, 8 dims

  // The part of a sequence that is worked on: blocks ``from`` .. ``to`` - 1 of n
  struct Part {
    int seq, pos, n, from, to, lo;
    int range, left;      // of the step's ranges; blocks up to its end
    int at, kvh, h0, heads;  // of the workgroups of the same keys: its key head, its query heads
    bool goes_on;         // it is not its range's first one
    Blocks blocks;
    const const_int* pages;
  };
  auto part_of = [&](Part p, int seq, int len, int from, int left) {
    p.seq = seq;
    p.pos = len - 1;
    p.blocks = visible_blocks(a, p.pos);
    p.n = p.blocks.n;
    p.from = from;
    p.to = min(p.n, from + left);
    p.left = left;
    p.lo = first_key(a, p.pos);
    p.pages = (const const_int*)(a.tables + (int64_t)seq * a.max_blocks);
    return p;
  };
  auto aim = [&](Part& p, int at) {
    p.at = at;
    p.kvh = per > 1 ? at / per : at;
    p.h0 = p.kvh * group + (at - p.kvh * per) * GM;
    p.heads = min(GM, group - (at - p.kvh * per) * GM);
  };
  Part p = {};  // that the loads are in
  aim(p, first_at);
  Cut cut = {};
  int done = 0;  // blocks of the workgroup's ranges ahead of this part
  if (CUT) {
    const Stretch x = find_range(a, -1, item, cut);
    if (x.seq < 0) return;  // more workgroups than there is work for
    p.range = item * cut.count;
    p = part_of(p, x.seq, x.len,
                cut.aligned ? (item - x.before) * cut.each : p.range * cut.each - x.before, cut.each);
  } else {
    p = part_of(p, item, a.seq_lens[item], 0, 1 << 30);
  }
  // The next part: of the next sequence, or of the next range, whose keys are of the workgroup's other head.
  // false: there is none
  auto go_on = [&]() {
    if (!RANGES || cut.aligned) return false;
    const int blocks = max(1, p.to - p.from);
    done += blocks;
    const int left = p.left - blocks;
    const bool same = left > 0, stays = !same && p.to < p.n;
    if (!same) {
      ++p.range;
      aim(p, p.at ^ 1);
      if (cut.count == 1 || !(p.range & 1)) return false;
    }
    const int seq = p.seq + !stays;
    if (seq >= a.seqs) return false;
    p.goes_on = same;
    p = part_of(p, seq, stays ? p.pos + 1 : ((const const_int*)a.seq_lens)[seq], stays ? p.to : 0,
                same ? left : cut.each);
    return true;
  };

  const uint32_t k_row = (uint32_t)a.G * D * 2, v_row = (uint32_t)a.G * V * 2;  // bytes
  const char* const k0 = (const char*)a.k_cache;
  const char* const v0 = (const char*)a.v_cache;
  const int shift = __builtin_ctz(a.kv_block);
  // Sequences that begin alike hold the same pages, at the same places of their tables.  Lanes look
  // at the next 64 sequences' page where this piece begins; a block whose pages are those of one that
  // has it too is left in the caches, others pass by them, as do not those that another workgroup of
  // the same key head reads.  All kept, all past, and so, us: 190 x 700 to 1300 keys of 8 heads, 608
  // in common 107, 117, 103, none 147, 133, 134; 60 of 32 heads 121, 131, 115 and 184, 168, 167; 16
  // heads a key head 64 x 700 to 1300 114, 121, 107.
  const const_int* others = p.pages;
  bool begins_alike = false;
  auto look = [&](int page, int there) {
    const uint64_t alike = __ballot(page == there && lane + 1 < a.seqs);
    begins_alike = alike != 0;
    int other = p.seq + 1 + (alike ? __builtin_ctzll(alike) : 0);
    if (other >= a.seqs) other -= a.seqs;
    others = (const const_int*)(a.tables + (int64_t)(begins_alike ? other : p.seq) * a.max_blocks);
  };
  struct Place {
    int slot[2];  // of a block's two groups of 16 keys
    int kvh;
    bool shared;
  };
  auto find = [&](int i) {
    Place at;
    at.kvh = p.kvh;
    const int key0 = p.blocks.key(i);
    auto key = [&](int g) { return min(key0 + 16 * g, p.pos & ~15); };
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int k = key(g);
      at.slot[g] = PAGED ? (p.pages[k >> shift] << shift) + (k & (a.kv_block - 1)) : 0;
    }
    at.shared = PAGED && begins_alike && p.pages[key(0) >> shift] == others[key(0) >> shift] &&
                p.pages[key(1) >> shift] == others[key(1) >> shift];
    return at;
  };
  // A load of keys has 8 rows of whole lines, 64 dims: the upper 8 rows of a product, and its upper 8
  // columns for the queries, have a line's other half.  Of its results those count whose row and
  // column have the same half; the halves' sums meet across lanes.
  constexpr int LINES = STEPS / 2;
  struct Rows {
    bf16x8_v k[2][2][LINES], v[NV];
  };
  const int c8 = c & 7, half = c >> 3;
  const uint32_t k_off = c8 * k_row + half * 64 + j * 16, v_off = kl * v_row + el * 16;
  auto load_paged = [&](auto shared, const Place& at, Rows& r) {
    const char* const kp = k0 + at.kvh * D * 2;
    const char* const vp = v0 + at.kvh * V * 2;
    auto get = [&](const char* p) {
      if constexpr (decltype(shared)::value) return *(const bf16x8_v*)p;
      return __builtin_nontemporal_load((const bf16x8_v*)p);
    };
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int s = 0; s < LINES; ++s)
          r.k[g][p][s] =
              get(kp + (uint64_t)(uint32_t)at.slot[g] * k_row + p * 8 * k_row + k_off + s * 128);
#pragma unroll
    for (int n = 0; n < NV; ++n)
      r.v[n] = get(vp + (uint64_t)(uint32_t)at.slot[n * KPL / 16] * v_row + n * KPL % 16 * v_row + v_off);
  };
  auto load = [&](int i, const Place& at, Rows& r) {
    if constexpr (PAGED) {
      // the comments keep the compiler from making one load of both kinds, which loses the hint
      if (per > 1 || at.shared) {
        asm volatile("; kept" ::: "memory");
        load_paged(std::true_type(), at, r);
        asm volatile("; kept, end" ::: "memory");
      } else {
        asm volatile("; past" ::: "memory");
        load_paged(std::false_type(), at, r);
        asm volatile("; past, end" ::: "memory");
      }
    } else {
      const int k = min(p.blocks.key(i) + (lane & (KB - 1)), p.pos), kvh = p.kvh;
      const int page = k / a.kv_block;
      if (lane < KB)
        slots[wid][lane] = a.tables[(int64_t)p.seq * a.max_blocks + page] * a.kv_block + k -
                           page * a.kv_block;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const uint32_t slot = slots[wid][g * 16 + p * 8 + c8];
          const char* kr = k0 + kvh * D * 2 + (uint64_t)slot * k_row + half * 64 + j * 16;
#pragma unroll
          for (int s = 0; s < LINES; ++s) r.k[g][p][s] = *(const bf16x8_v*)(kr + s * 128);
        }
#pragma unroll
      for (int n = 0; n < NV; ++n)
        r.v[n] = *(const bf16x8_v*)(v0 + kvh * V * 2 + (uint64_t)(uint32_t)slots[wid][n * KPL + kl] * v_row +
                                    el * 16);
      __builtin_amdgcn_wave_barrier();
    }
  };
  // A part's first loads: the workgroup's blocks go to the waves in turn, whichever sequences they are of.
  // The heads' queries are columns, 8 dims a lane and step
  Rows r0, r1;
  Place at{};
  int i;
  bf16x8_v q[LINES];
  auto begin = [&]() {
    i = p.from + ((wid - done) & 3);
    if (i < p.to) {
      // a part of a few blocks is over before the answer pays
      const bool ask = PAGED && per == 1 && a.seqs > 1 && p.to - p.from > 8;
      int there = 0;
      const int first = min(p.blocks.key(p.from), p.pos & ~15) >> shift;
      if (ask) {
        int other = p.seq + 1 + lane;
        other -= other >= a.seqs ? a.seqs : 0;
        there = a.tables[(int64_t)min(other, a.seqs - 1) * a.max_blocks + first];
      }
      begins_alike = false;
      load(i, find(i), r0);
      if (ask) look(p.pages[first], there);
      if (AHEAD && PAGED) at = find(min(i + 4, p.n - 1));
    }
    const int head = p.h0 + min(c8, p.heads - 1);
#pragma unroll
    for (int s = 0; s < LINES; ++s)
      q[s] = *(const bf16x8_v*)((const bf16_t*)a.q + p.seq * a.q_stride + (int64_t)head * D +
                                s * 64 + half * 32 + j * 8);
  };
  begin();

  // scores in the exp2 domain: a factor, or c1 - 2 c1 / (exp2(c3 s) + 1)
  const float c1 = a.cap * LOG2E;
  const float mul = a.cap > 0.f ? 2.f * LOG2E * a.scale / a.cap : a.scale * LOG2E;
  float m, l;
  // biases: distances of n_bias - 1 and more share one
  const int far = a.n_bias - 1;
  const float* bias = nullptr;
  float b_far = 0.f;
  float acc[GM][8];
  auto barrier = [&]() {  // of LDS alone: loads stay under way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  auto work = [&](int i, Rows& r) {
    const int key0 = p.blocks.key(i), pos = p.pos, lo = p.lo;
    auto hidden = [&](int key) { return (key > pos) | ((key < lo) & (key >= a.keep)); };
    f32x4_v halves[2][2] = {}, s[2];
#pragma unroll
    for (int st = 0; st < LINES; ++st)
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          halves[g][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.k[g][p][st], q[st],
                                                                 halves[g][p], 0, 0, 0);
    // lanes of columns below 8: 4 keys of their row group, as of a product of 16 keys
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto of = __builtin_amdgcn_permlane32_swap(__float_as_int(halves[g][0][e]),
                                                         __float_as_int(halves[g][1][e]), false, false);
        const int upper = __builtin_amdgcn_update_dpp(0, of[1], 0x128, 0xf, 0xf, false);  // row_ror:8
        s[g][e] = __int_as_float(of[0]) + __int_as_float(upper);
      }
    float w[8], mt = NEG;
    const bool edge = key0 + KB - 1 > pos || (key0 < lo && key0 + KB > a.keep);
    const bool near = bias && pos - (key0 + KB - 1) < far;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int key = key0 + (e >> 2) * 16 + 4 * j + (e & 3);
      float x = s[e >> 2][e & 3] * mul;
      if (a.cap > 0.f) x = c1 - 2.f * c1 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
      x += near ? bias[min(max(pos - key, 0), far)] * LOG2E : b_far;
      if (edge && hidden(key)) x = -INFINITY;
      w[e] = x;
      mt = fmaxf(mt, x);
    }
    if (edge) {  // what no token has written may be anything
#pragma unroll
      for (int n = 0; n < NV; ++n)
        if (hidden(key0 + n * KPL + kl)) r.v[n] = bf16x8_v{};
    }
    if constexpr (SIG) {
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-w[e]));
    } else {
      mt = max_with<32>(max_with<16>(mt));
      if (__any(c < 8 && mt > m)) {
        const float up = fmaxf(m, mt), alpha = __builtin_amdgcn_exp2f(m - up);
        m = up;
        l *= alpha;
        if (lane < GM) rescale[wid][lane] = alpha;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int g = 0; g < GM; ++g) {
          const float f = rescale[wid][g];
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[g][e] *= f;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        w[e] = __builtin_amdgcn_exp2f(w[e] - m);
        l += w[e];
      }
    }
    if (c < GM)
#pragma unroll
      for (int e = 0; e < 8; ++e) weight[wid][(e >> 2) * 16 + 4 * j + (e & 3)][c] = w[e];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      float f[GM];
#pragma unroll
      for (int g = 0; g < GM; ++g) f[g] = weight[wid][n * KPL + kl][g];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = (float)r.v[n][e];
#pragma unroll
        for (int g = 0; g < GM; ++g) acc[g][e] += f[g] * v;
      }
    }
    __builtin_amdgcn_wave_barrier();
  };
  for (;;) {
    const int head = p.h0 + min(c8, p.heads - 1);
    if (a.bias) {
      bias = a.bias + (int64_t)head * a.n_bias;
      b_far = bias[far] * LOG2E;
    }
    const bool sink = a.sink && p.from == 0 && wid == 0;
    m = sink ? a.sink[head] * LOG2E : NEG;
    l = sink && j == 0 ? 1.f : 0.f;
#pragma unroll
    for (int g = 0; g < GM; ++g)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;
    if constexpr (AHEAD) {
      for (; i < p.to; i += 8) {
        if (i + 4 < p.to) {
          load(i + 4, at, r1);
          if (PAGED) at = find(min(i + 8, p.n - 1));
        }
        work(i, r0);
        if (i + 4 >= p.to) break;
        if (i + 8 < p.to) {
          load(i + 8, at, r0);
          if (PAGED) at = find(min(i + 12, p.n - 1));
        }
        work(i + 4, r1);
      }
    } else {
      for (; i < p.to; i += 4) {
        work(i, r0);
        if (i + 4 < p.to) load(i + 4, find(i + 4), r0);
      }
    }

    // where the results go, and the next part, whose first loads run meanwhile
    const int seq = p.seq, slot = 2 * p.range + (p.to < p.n && p.goes_on);
    const int h0 = p.h0, heads = p.heads;
    const bool whole = p.from == 0 && p.to == p.n, more = go_on();
    if (RANGES && more) begin();
    // the lanes with the same dims, then the waves
    l = sum_with<32>(sum_with<16>(l));
    if (lane < GM) lds_ml[wid][lane] = float2{m, l};
#pragma unroll
    for (int g = 0; g < GM; ++g)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float o = acc[g][e];
        if (LPK <= 8) o = sum_with<8>(o);
        if (LPK <= 16) o = sum_with<16>(o);
        o = sum_with<32>(o);
        if (lane < LPK) lds_acc[wid][g][el * 8 + e] = o;
      }
    barrier();
    for (int n = threadIdx.x; n < heads * V; n += 256) {
      const int g = n / V, e = n % V;
      float mx = NEG, sum = 0.f, o = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) mx = fmaxf(mx, lds_ml[w][g].x);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float f = SIG ? 1.f : __builtin_amdgcn_exp2f(lds_ml[w][g].x - mx);
        sum += f * lds_ml[w][g].y;
        o += f * lds_acc[w][g][e];
      }
      if (whole) {
        if (!SIG) o = sum > 0.f ? o / sum : 0.f;
        if (a.gate) o *= sigmoid_f(bf2f(((const bf16_t*)a.gate)[seq * a.gate_stride + h0 + g]));
        ((bf16_t*)a.out)[seq * a.out_stride + (int64_t)(h0 + g) * V + e] = from_f<bf16_t>(o);
      } else {
        const int64_t row = (int64_t)slot * a.H + h0 + g;
        a.part[row * V + e] = o;
        if (e == 0) a.part_ml[row] = float2{mx, sum};
      }
    }
    if (!RANGES || !more) break;
    barrier();
  }
}

// Sequences and workgroups of the same keys from which ranges are the faster cut, us with the merge: of 8 key heads
// 1 x 4001 keys 13.9 by pieces and 14.4, 12 x 150 to 980 16.5 and 17.5, 16 x 350 to 1000 21.0 and 21.9, 20 x 130 to
// 3900 45.5 and 45.0, 24 x 510 to 2400 43.5 and 41.0; of 32, 3 x 850 to 2700 28.6 and 29.0, 6 x 720 to 3800 49.7
// and 49.1
#define RANGES_FROM 160

// Merge the pieces of the rows: a lane has 4 dims of a head.  Workgroups are few, so that those
// with nothing to merge cost little: one wave each up to MERGE_ROWS rows, else 4.
#define MERGE_ROWS 1024
template <int VN, bool SIG>
__global__ __launch_bounds__(256) void merge_pieces_kernel(const GroupedArgs a) {
  constexpr int V = 64 * VN, LANES = V / 4;  // lanes a head
  const int at = blockIdx.x * blockDim.x + threadIdx.x;
  const int h = min(at / LANES, a.H - 1), e = at % LANES * 4, seq = blockIdx.y;
  Cut cut;
  const Stretch x = find_range(a, seq, 0, cut);
  int first = x.before, pieces, ahead = 0;
  if (cut.aligned) {
    pieces = x.n;
  } else {
    first = quotient(x.before, cut.each);
    pieces = quotient(x.before + x.n - 1, cut.each) - first + 1;
    // a range's part of a sequence that goes on is its second one if another sequence is ahead of it
    ahead = first * cut.each < x.before;
  }
  if (pieces == 1) return;  // written by the workgroup
  auto row_of = [&](int i) { return (int64_t)(2 * (first + i) + (i == 0 && ahead)) * a.H + h; };
  float m = NEG, l = 0.f, o[4] = {};
  if (!SIG) {
    // maxima and sums, a lane each
    for (int i = e / 4; i < pieces; i += LANES) m = fmaxf(m, a.part_ml[row_of(i)].x);
#pragma unroll
    for (int off = LANES / 2; off; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    for (int i = e / 4; i < pieces; i += LANES) {
      const float2 ml = a.part_ml[row_of(i)];
      l += ml.y * __builtin_amdgcn_exp2f(ml.x - m);
    }
#pragma unroll
    for (int off = LANES / 2; off; off >>= 1) l += __shfl_xor(l, off, 64);
  }
#pragma unroll 8
  for (int i = 0; i < pieces; ++i) {
    const int64_t row = row_of(i);
    const float w = SIG ? 1.f : __builtin_amdgcn_exp2f(a.part_ml[row].x - m);
    const float4 v = *(const float4*)(a.part + row * V + e);
    o[0] += w * v.x;
    o[1] += w * v.y;
    o[2] += w * v.z;
    o[3] += w * v.w;
  }
  if (at / LANES >= a.H) return;
  float by = SIG ? 1.f : l > 0.f ? 1.f / l : 0.f;
  if (a.gate) by *= sigmoid_f(bf2f(((const bf16_t*)a.gate)[seq * a.gate_stride + h]));
#pragma unroll
  for (int n = 0; n < 4; ++n) o[n] *= by;
  store_f<4>((bf16_t*)a.out + seq * a.out_stride + (int64_t)h * V + e, o);
}

// Any dtype and size: a workgroup per (token, head), its 4 waves stride over the keys,
// a lane holds every 64th dim.
template <typename T, int NE>
__global__ __launch_bounds__(256) void grouped_plain_kernel(
    const GroupedArgs a, const int d, const int v) {
  const int h = blockIdx.y, kvh = h / (a.H / a.G);
  int seq, pos, token;
  if (a.tile_seq) {
    seq = a.tile_seq[blockIdx.x];
    pos = a.ctx_lens[seq] + a.tile_q0[blockIdx.x];
    token = a.row_starts[seq] + a.tile_q0[blockIdx.x];
  } else {
    seq = token = blockIdx.x;
    pos = a.seq_lens[seq] - 1;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int* table = a.tables + (int64_t)seq * a.max_blocks;
  const T* qr = (const T*)a.q + token * a.q_stride;
  float q[NE], acc[NE] = {};
  // mixed scores are those of one long query, the mix of the heads that share a key head,
  // against all key heads
  const int dk = a.talk ? a.G * d : d, k_at = a.talk ? 0 : kvh * d, group = a.H / a.G;
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int i = e * 64 + lane;
    q[e] = 0.f;
    if (i >= dk) continue;
    if (a.talk) {
      const int g0 = i / d * group;
      for (int g = g0; g < g0 + group; ++g)
        q[e] += a.talk[h * a.H + g] * to_f(qr[(int64_t)g * d + i % d]);
    } else {
      q[e] = to_f(qr[(int64_t)h * d + i]);
    }
  }
  const bool sink = a.sink && wid == 0;
  float m = sink ? a.sink[h] : NEG, l = sink ? 1.f : 0.f;
  const KeyList keys = visible_keys(a, pos);
  for (int x = wid; x < keys.n; x += 4) {
    const int k = keys.at(x);
    const int64_t slot = (int64_t)table[k / a.kv_block] * a.kv_block + k % a.kv_block;
    const T* kr = (const T*)a.k_cache + slot * a.G * d + k_at;
    const T* vr = (const T*)a.v_cache + (slot * a.G + kvh) * v;
    float dot = 0.f, val[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int i = e * 64 + lane;
      if (i < dk) dot += q[e] * to_f(kr[i]);
      val[e] = i < v ? to_f(vr[i]) : 0.f;
    }
    dot = wave_sum(dot) * a.scale;
    if (a.cap > 0.f) dot = a.cap * tanhf(dot / a.cap);
    if (a.bias) dot += a.bias[(int64_t)h * a.n_bias + min(pos - k, a.n_bias - 1)];
    if (a.sigmoid) {
      const float p = 1.f / (1.f + expf(-dot));
#pragma unroll
      for (int e = 0; e < NE; ++e) acc[e] += p * val[e];
      continue;
    }
    const float mn = fmaxf(m, dot);
    const float alpha = expf(m - mn), p = expf(dot - mn);
    m = mn;
    l = l * alpha + p;
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[e] = acc[e] * alpha + p * val[e];
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
    w[i] = a.sigmoid ? 1.f : expf(ml[i].x - mx);
    sum += w[i] * ml[i].y;
  }
  float f = a.sigmoid ? 1.f : 1.f / sum;
  if (a.gate) f *= sigmoid_f(to_f(((const T*)a.gate)[token * a.gate_stride + h]));
  for (int i = threadIdx.x; i < v; i += 256) {
    float o = 0.f;
#pragma unroll
    for (int n = 0; n < 4; ++n) o += w[n] * part[n][i];
    ((T*)a.out)[token * a.out_stride + (int64_t)h * v + i] = from_f<T>(o * f);
  }
}

// k [n, G, d] and v [n, G, v] rows into their slots, 16 bytes a thread.
__global__ __launch_bounds__(256) void cache_keys_values_kernel(
    ulonglong2* __restrict__ k_cache, ulonglong2* __restrict__ v_cache,
    const ulonglong2* __restrict__ k, const ulonglong2* __restrict__ v,
    const int64_t* __restrict__ slots, const int k_units, const int v_units,
    const int64_t stride, const int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int units = k_units + v_units;
  const int64_t n = i / units;
  const int u = (int)(i - n * units);
  if (u < k_units)
    k_cache[slots[n] * k_units + u] = k[n * stride + u];
  else
    v_cache[slots[n] * v_units + u - k_units] = v[n * stride + u - k_units];
}

template <int DN, int VN, int GM, bool SIG>
static void launch_decode(const GroupedArgs& a, hipStream_t stream) {
  const int per = a.G * ((a.group + GM - 1) / GM);
  const int items = a.ranges ? a.pieces : a.pieces ? 2 * a.pieces + a.seqs : a.seqs, grid = items * per;
  const bool paged = a.kv_block >= 16 && (a.kv_block & (a.kv_block - 1)) == 0;
  auto kernel = paged ? a.pieces ? grouped_decode_kernel<DN, VN, GM, SIG, true, true, false>
                                 : grouped_decode_kernel<DN, VN, GM, SIG, true, false, false>
                : a.pieces ? grouped_decode_kernel<DN, VN, GM, SIG, false, true, false>
                           : grouped_decode_kernel<DN, VN, GM, SIG, false, false, false>;
  if constexpr (GM < 8)
    if (a.ranges)
      kernel = paged ? grouped_decode_kernel<DN, VN, GM, SIG, true, true, true>
                     : grouped_decode_kernel<DN, VN, GM, SIG, false, true, true>;
  kernel<<<grid, 256, 0, stream>>>(a);
}

template <int DN, int VN>
static bool launch_decode(const GroupedArgs& args, int gm, hipStream_t stream) {
  GroupedArgs a = args;
  a.gm = gm;
  a.shared_from = DN + VN <= 4 ? 16 : 12;
  a.ranges = a.pieces && gm < 8 && a.seqs * a.G * ((a.group + gm - 1) / gm) >= RANGES_FROM;
  if (gm == 1)
    (a.sigmoid ? launch_decode<DN, VN, 1, true> : launch_decode<DN, VN, 1, false>)(a, stream);
  else if (gm == 2)
    (a.sigmoid ? launch_decode<DN, VN, 2, true> : launch_decode<DN, VN, 2, false>)(a, stream);
  else if (gm == 4)
    (a.sigmoid ? launch_decode<DN, VN, 4, true> : launch_decode<DN, VN, 4, false>)(a, stream);
  else if (gm == 8)
    (a.sigmoid ? launch_decode<DN, VN, 8, true> : launch_decode<DN, VN, 8, false>)(a, stream);
  else
    return false;
  if (a.pieces == 0) return true;
  auto merge = a.sigmoid ? merge_pieces_kernel<VN, true> : merge_pieces_kernel<VN, false>;
  const int threads = a.H * a.seqs <= MERGE_ROWS ? 64 : 256, lanes = a.H * 16 * VN;
  merge<<<dim3((lanes + threads - 1) / threads, a.seqs), threads, 0, stream>>>(a);
  return true;
}

template <int DN>
static bool launch_decode_v(const GroupedArgs& a, int v, int gm, hipStream_t stream) {
  switch (v) {
    case 64: return launch_decode<DN, 1>(a, gm, stream);
    case 128: return launch_decode<DN, 2>(a, gm, stream);
    case 256: return launch_decode<DN, 4>(a, gm, stream);
    default: return false;
  }
}

template <typename T>
static bool launch_plain(const GroupedArgs& a, int d, int v, int tokens, hipStream_t stream) {
  const int dk = a.talk ? a.G * d : d;
  const int ne = ((dk > v ? dk : v) + 63) / 64;
  if (ne > 64) return false;
  auto k = ne <= 1    ? grouped_plain_kernel<T, 1>
           : ne <= 2  ? grouped_plain_kernel<T, 2>
           : ne <= 4  ? grouped_plain_kernel<T, 4>
           : ne <= 8  ? grouped_plain_kernel<T, 8>
           : ne <= 32 ? grouped_plain_kernel<T, 32>
                      : grouped_plain_kernel<T, 64>;
  k<<<dim3(tokens, a.H), 256, 0, stream>>>(a, d, v);
  return true;
}

extern "C" {

// gm: query heads of one key/value head per workgroup, 1, 2, 4 or 8
bool launch_grouped_decode(const GroupedArgs* a, int d, int v, int gm, hipStream_t stream) {
  switch (d) {
    case 64: return launch_decode_v<1>(*a, v, gm, stream);
    case 128: return launch_decode_v<2>(*a, v, gm, stream);
    case 256: return launch_decode_v<4>(*a, v, gm, stream);
    default: return false;
  }
}

bool launch_grouped_plain(bool bf16, const GroupedArgs* a, int d, int v, int tokens,
                          hipStream_t stream) {
  return (bf16 ? launch_plain<bf16_t> : launch_plain<float>)(*a, d, v, tokens, stream);
}

void launch_cache_keys_values(void* k_cache, void* v_cache, const void* k, const void* v,
                              const int64_t* slots, int k_units, int v_units, int64_t stride,
                              int n, hipStream_t stream) {
  const int64_t total = (int64_t)n * (k_units + v_units);
  cache_keys_values_kernel<<<(total + 255) / 256, 256, 0, stream>>>(
      (ulonglong2*)k_cache, (ulonglong2*)v_cache, (const ulonglong2*)k,
      (const ulonglong2*)v, slots, k_units, v_units, stride, total);
}

}  // extern "C"
