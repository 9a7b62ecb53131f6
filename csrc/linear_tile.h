// The tiles of linear.hip's and experts_gemm.hip's products (device code).
#pragma once
#include <type_traits>

#include "common_t.h"
#include "gated_act.h"
#include "linear.h"

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;

// Where a piece of work is: rows m0 .. m1 - 1, first output, chunks of the inner dimension, its number
// among the parts of that, w, x with as many rows, what its Work adds to rows, the chunk that it
// begins with where linear_tiles() takes them in turn
struct LinearSpot {
  int m0, m1, o0, first, last, part;
  const void *w, *x;
  int x_rows, row0, at;
};

// n / (1 + exp(-z)), the same bits as the division's for all n of 16 bits, in fewer instructions: a
// quarter of the divisor has a reciprocal at all its sizes and needs no scaling.  The reciprocal is
// one ulp off before a Newton step, the quotient takes in its remainder (Markstein's way), and the
// hardware puts infinities and what is no number right.  The unit ends a tile of products and nothing
// else runs beside it: 15675 x 28672 x 4096 SwiGLU takes 1.8% longer than with the reciprocal
// alone, by the division 2.7%.
DEV float by_sigmoid(float n, float z) {
  const float d = __builtin_fmaf(__expf(-z), 0.25f, 0.25f), n4 = 0.25f * n;
  float r = __builtin_amdgcn_rcpf(d);
  r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
  const float q = n4 * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, n4), r, q), d, n4);
}

// The gated unit of two sums, both rounded first, as they are between two passes
template <int UNIT>
DEV float unit_of(const LinearArgs& a, float gate, float up) {
  gate = (float)(__bf16)gate;
  up = (float)(__bf16)up;
  if (UNIT == LINEAR_SWIGLU) return by_sigmoid(gate, gate) * up;
  gate = fminf(gate, a.limit);
  float z = a.alpha * gate;
  if (a.cubic != 0.f) z *= 1.f + a.cubic * gate * gate;
  return gate * by_sigmoid(1.f, z) * (fminf(fmaxf(up, -a.limit), a.limit) + a.offset);
}

#ifdef __HIP_DEVICE_COMPILE__  // the host knows no buffer resources
// Works start, start + step .. below total of a workgroup of 4 waves.  Fragments of a wave along
// the outputs (FN) and the rows (FM); chunks of w (WS) and x (XS) in LDS.  ONCE: no other
// workgroup reads the same weights, whose loads then pass by the caches (nt), and the chunks of a work
// that is no part are taken in turn from its spot's ``at`` on.
template <int FN, int FM, int WS, int XS, int UNIT, bool ONCE = false, class Work>
DEV void linear_tiles(const LinearArgs& a, const Work& work, char* const lds) {
  constexpr bool GLU = UNIT == LINEAR_SWIGLU || UNIT == LINEAR_GLU;
  constexpr bool TURNS = ONCE && UNIT != LINEAR_PARTS;
  constexpr int TN = 32 * FN, TM = 32 * FM;    // rows of w and of x of a tile
  constexpr int LW = FN, LX = FM;              // a wave's loads of a chunk, 8 rows each
  constexpr int SW = TN * 128, SX = TM * 128;  // a chunk's bytes
  constexpr int NM = FN * FM;
  // loads behind a chunk's last one when it is waited for
  constexpr int BEHIND = XS < WS ? LW + (XS - 2) * (LW + LX) : (WS - 2) * (LW + LX);
  static_assert(BEHIND < 64 && XS >= 2 && WS >= 3);
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wid & 1, wm = wid >> 1;
  const int c = lane & 15, g = lane >> 4;
  const int outs = GLU ? a.N / 2 : a.N;
  auto buffer = [](const void* p, int64_t rows, int64_t stride, int64_t row) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(((rows - 1) * stride + row) * 2),
                                             0x00020000);
  };
  auto bx = buffer(a.x, 1, 0, 0), bw = buffer(a.w, 1, 0, 0);  // of the cursors' works
  const int slot = ((lane & 7) ^ (lane >> 3)) * 16;
  int vw[LW], vx[LX];  // this lane's rows
  // cursors of the loads: work, chunk, its last one, place in LDS; past the last work its
  // chunks again.  In turn: the chunks left
  int tw = work.start, cw, ew, w0, nw = 0, sw = 0;
  int tx = work.start, cx, ex, x0, nx = 0, sx = 0;
  auto aim_w = [&](int t) {
    const LinearSpot spot = work.spot(t);
    cw = TURNS ? spot.at : spot.first;
    ew = spot.last;
    w0 = spot.first;
    if (TURNS) nw = ew - w0;
    bw = buffer(spot.w, a.N, a.w_stride, a.K);
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      // in such an order that a lane's sums are of 8 neighbours
      const int p = (wid * LW + i) * 8 + (lane >> 3), f = p >> 4, k = p & 15;
      const int in = 8 * (k >> 2) + 4 * (f & 1) + (k & 3);
      int o = min(spot.o0 + (GLU ? f >> 2 : f >> 1) * 32 + in, outs - 1);
      if (GLU && (f & 2)) o += outs;
      vw[i] = (int)(o * a.w_stride) * 2 + slot;
    }
  };
  auto aim_x = [&](int t) {
    const LinearSpot spot = work.spot(t);
    cx = TURNS ? spot.at : spot.first;
    ex = spot.last;
    x0 = spot.first;
    if (TURNS) nx = ex - x0;
    bx = buffer(spot.x, spot.x_rows, a.x_stride, a.K);
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int p = (wid * LX + i) * 8 + (lane >> 3);
      vx[i] = (int)(work.x_row(spot, min(spot.m0 + p, spot.m1 - 1)) * a.x_stride) * 2 + slot;
    }
  };
  auto load_w = [&](int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(bw, (lds_char*)(lds + sw + (wid * LW + i) * 1024), 16,
                                             vw[i], cw * 128, 0, ONCE ? 2 : 0);
  };
  auto load_x = [&](int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        bx, (lds_char*)(lds + WS * SW + sx + (wid * LX + i) * 1024), 16, vx[i], cx * 128, 0, 0);
  };
  auto next_w = [&]() {
    sw = sw == (WS - 1) * SW ? 0 : sw + SW;
    ++cw;
    const bool end = TURNS ? --nw == 0 : cw == ew;
    if (cw == ew) cw = w0;
    if (end) {
      const int t = work.next(tw);
      if (t != tw)
        aim_w(tw = t);
      else if (TURNS)
        nw = ew - w0;
    }
  };
  auto next_x = [&]() {
    sx = sx == (XS - 1) * SX ? 0 : sx + SX;
    ++cx;
    const bool end = TURNS ? --nx == 0 : cx == ex;
    if (cx == ex) cx = x0;
    if (end) {
      const int t = work.next(tx);
      if (t != tx)
        aim_x(tx = t);
      else if (TURNS)
        nx = ex - x0;
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
  for (int k = 0; k < (WS - 1 > XS ? WS - 1 : XS); ++k) {
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
  // The first chunk has landed.  To wait for the whole rings, as was done, has the memory run idle once
  // while no loads follow them, us of products alone: 40 x 2048 x 2048 9.4 and now 8.7, 61 x 4096 x
  // 4096 14.0 and 13.4, 61 x 28672 x 4096 SwiGLU 38.6 and 38.1; experts of 4093 tokens 1010 and 1000
  constexpr int STARTED = (WS - 2) * LW + (XS - 1) * LX;
  static_assert(STARTED < 64);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STARTED) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  look(0);
#pragma unroll
  for (int i = 0; i < FN + FM; ++i) read(0, i);

  for (int t = work.start; t < work.total; t += work.step) {
    const LinearSpot spot = work.spot(t);
    const int m0 = spot.m0, o0 = spot.o0;
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
    for (int k = spot.last - spot.first; k > 1; --k) chunk(std::false_type());

    // sums r of fragments i (and i + 1) and j: row c of 16, outputs 8 g + r (and 4 + r) of 32
    constexpr int GROUP = GLU ? 4 : 2;  // fragments of 32 outputs
    if (UNIT == LINEAR_PARTS) {
      float* const sums = (float*)a.out + spot.part * (int64_t)a.M * a.N;
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const int m = m0 + (wm * FM + j) * 16 + c;
        if (m >= spot.m1) continue;
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
    if (Work::ANY_WIDTH && (outs & 7)) {  // no rows of 16-byte units
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const int m = m0 + (wm * FM + j) * 16 + c;
        if (m >= spot.m1) continue;
        __bf16* const to = out + work.out_row(spot, m) * a.out_stride;
#pragma unroll
        for (int i = 0; i < FN; i += GROUP) {
          const int o = o0 + (wn * (FN / GROUP) + i / GROUP) * 32 + 8 * g;
          const bf16x8_v v = __builtin_bit_cast(bf16x8_v, eight(i, j, o));
#pragma unroll
          for (int r = 0; r < 8; ++r)
            if (o + r < outs) to[o + r] = v[r];
        }
      }
      continue;
    }
    const bool low = c < 8;
    constexpr bool PAIRS = FN >= 2 * GROUP;
    int64_t rows[FM][2];  // all asked for before the first is needed
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int m = m0 + (wm * FM + j) * 16 + (PAIRS ? (c & 7) + 8 * h : c);
        if (!h || PAIRS) rows[j][h] = work.out_row(spot, min(m, spot.m1 - 1)) * a.out_stride;
      }
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
          if (oo < outs) {
            if (mm < spot.m1)
              __builtin_nontemporal_store(upper, (u32x4_v*)(out + rows[j][0] + oo));
            if (mm + 8 < spot.m1)
              __builtin_nontemporal_store(lower, (u32x4_v*)(out + rows[j][1] + oo));
          }
        } else if (m + c < spot.m1 && o < outs) {
          const int64_t row = PAIRS ? work.out_row(spot, m + c) * a.out_stride : rows[j][0];
          __builtin_nontemporal_store(p, (u32x4_v*)(out + row + o));
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end
}
#endif
