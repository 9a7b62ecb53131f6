// The gated delta rule of a prompt by chunks of 16 tokens on the fp32 matrix cores (gfx950): bf16 inputs,
// heads with 128 key channels, values of whole 16s.
//
// Within a chunk, with P_i the decays' product up to token i, S0 the state ahead of it and
// A_ij = sum_d k_i k_j P_i / P_j, B_ij the same with q_i:
//   u = M (v - (P k)^T S0),  M = (I + beta A)^-1 beta    A below the diagonal
//   o = (P q)^T S0 + B u                                 B with the diagonal
//   S = P_15 S0 + sum_i (P_15 / P_i) k_i u_i^T
// M, B and the scaled q and k do not depend on the state.  So a chain of four steps a chunk is left, products
// of the 128 channels by P k and P q, their sum over the waves, u, and the state's update, instead of
// 16 reductions.
//
// Everything is fp32, as token by token.  All quotients of decays are products of decays between two
// tokens, by halves: pairs on both sides of a block's middle take the decays behind the middle on the
// one and ahead of it on the other side, so that nothing overflows or is divided.  M's entries are at most 1, as
// the updates I - beta k k^T do not grow anything; its rows cancel where keys are alike, so that it is solved in 64
// bits (by 96 registers 91 us a layer of 5 sequences, by the 140 that the compiler takes 99.6).
//
// States against 64 bits, 320 tokens, errors of norms by chunks over token by token: keys that are not alike 0.88 to
// 1.10 (the latter under decays of 0.7 a token, 0.7e-7 and 0.63e-7), keys of a product of 0.5 0.9 to 1.06, of 0.9
// 0.9 to 1.33 (1.2e-7 and 0.9e-7).  Results ahead of the norm, in which (P q)^T S0 and B u cancel, 0.95 to 1.1,
// 0.9 to 1.6 and 1.0 to 2.3 (2.4e-7 and 1.0e-7), which are rounded to 16 bits behind it.
//
//   delta_chunk_kernel: a workgroup a chunk and head: P k, P q, P_15 / P k, P_15, M and B, in the
//     order of the matrix cores' operands
//   delta_chunk_scan_kernel: a workgroup 16 CB columns of a head's state.  Each of 8 waves has 16
//     channels of it, as the result of its own update, which is the second operand of the next products
//     as it is; one wave of 16 columns adds up their products by P k and makes u, while they go on
//     with P q, and another one makes o, so that neither the chain nor u waits for loads or stores
//
// Bound by the chain of the longest sequence, 0.95 us a chunk and 16 columns (a fifth each the two
// kinds of products, the sums over the waves, the barriers and the update), or by the fp32 matrix cores.  16
// heads of 128 x 128, 5 sequences of 530 to 2370 tokens, us: token by token 519, in chunks 94 for their
// operands (192 MB written) and 209; 8000 tokens of one sequence, all launches, 1444 and 631.  4 waves of 32
// channels that each make u, with one barrier a chunk, were 7% faster for one sequence and 15% slower for
// several; u by W^T S0 with W = M (P k) made ahead loses digits of v.
#include "delta_device.h"
#include "launch.h"

typedef float f32x4_v __attribute__((ext_vector_type(4)));

// Floats of a chunk and head in the workspace: P k, P q, P_15 / P k; P_15; M, B
#define FRAG 2048
#define AT_DECAY (3 * FRAG)
#define AT_M (AT_DECAY + 128)
#define AT_B (AT_M + 256)
static_assert(AT_B + 256 == DELTA_CHUNK_FLOATS, "layout");

// Tokens are in the matrices' rows and inner elements so that a product's steps take them in order, four by four
// (lane group g has tokens g, 4 + g, 8 + g and 12 + g): what came last, which decays leave the largest, is added
// last.  In the order of the lanes' rows the states of random keys under decays of 0.7 a token were 1.25 to 1.5
// times as far from 64 bits as token by token (0.94e-7 and 0.63e-7), so 1.0 to 1.1 times.
DEV int place(int token) { return 4 * (token & 3) + (token >> 2); }  // and the token at a place

// A wave's 16 channels in the order that its products take them: position 4 g + r
DEV int channel_of(int wave, int g, int r) { return 32 * (wave >> 1) + 8 * g + 4 * (wave & 1) + r; }

DEV f32x4_v product(f32x4_v a, f32x4_v b, f32x4_v c) {  // 16 x 16 of 16 inner elements
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
#endif
  return c;
}

// product() by a lower triangle, c + a x, where x may hold what is no number, which must not reach the
// tokens ahead of it through the zeros of the upper triangle: then row by row
DEV f32x4_v causal(f32x4_v a, f32x4_v x, f32x4_v c) {
  f32x4_v y = product(a, x, c);
  const float sum = fabsf(x[0]) + fabsf(x[1]) + (fabsf(x[2]) + fabsf(x[3]));
  if (__ballot(!(sum < INFINITY))) {
    const int first = (threadIdx.x & 63) >> 4;
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {
      f32x4_v past;
#pragma unroll
      for (int r = 0; r < 4; ++r) past[r] = first + 4 * r <= i ? x[r] : 0.f;
      past = product(a, past, c);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = first + 4 * r == i ? past[r] : y[r];
    }
  }
  return y;
}

template <int CTRL>
DEV float dpp(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// In blocks of 2 H lanes: the upper half's lanes get the lower half's last value and the other way
// round
template <int H>
DEV float across(float v, bool upper) {
  if (H == 1) return dpp<0xb1>(v);                   // quad_perm 1 0 3 2
  if (H == 2) return dpp<0x5f>(v);                   // quad_perm 3 3 1 1
  if (H == 4) return dpp<0x141>(dpp<0xff>(v));       // quad_perm 3 3 3 3, row_half_mirror
  const float low = dpp<0x157>(v), high = dpp<0x15f>(v);  // row_newbcast 7, 15
  return upper ? low : high;
}

// grid (tiles of 16 tokens, H), 4 waves: wave w channels 32 w .. 32 w + 31, lane (token, 8 of them)
__global__ __launch_bounds__(256, 5) void delta_chunk_kernel(const DeltaArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  __shared__ f32x4_v sums[4][2][64];
  __shared__ float turn[4][16][36];
  const int tile = blockIdx.x, h = blockIdx.y, kvh = h / (a.H / a.G);
  const int seq = a.tile_seq[tile], q0 = a.tile_q0[tile];
  const int n = min(16, a.seq_lens[seq] - a.ctx_lens[seq] - q0);
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4, d = 32 * wid + 8 * g;
  const int64_t first = a.row_starts[seq], row = first + q0 + min(m, n - 1);
  float* const ws = a.chunks + ((int64_t)h * (a.N / 16 + a.seqs) + first / 16 + seq + q0 / 16) *
                                   DELTA_CHUNK_FLOATS;

  // tokens past the end change nothing: decay 1, k = q = beta = 0
  const bool in = m < n;
  float q[8], k[8], F[8], E[8], beta, kq;
  {
    const bf16_t* y = (const bf16_t*)a.y + row * a.C + kvh * 128 + d;
    load_f<8>(q, y);
    load_f<8>(k, y + a.G * 128);
    if (!a.head_decay) load_f<8>(F, a.g + (row * a.H + h) * 128 + d);
    const float* unit = a.unit + (row * a.G + kvh) * 3;
    const float fq = unit[0], fk = unit[1];
    kq = in ? unit[2] : 0.f;
    beta = in ? sigmoid_f(to_f(((const bf16_t*)a.b)[row * a.b_stride + h])) : 0.f;
    if (a.head_decay) {
      const float z = to_f(((const bf16_t*)a.z)[row * a.z_stride + h]);
      F[0] = decay_f(z + a.dt_bias[h], expf(a.A_log[h]));
#pragma unroll
      for (int e = 1; e < 8; ++e) F[e] = F[0];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      q[e] = in ? q[e] * fq : 0.f;
      k[e] = in ? k[e] * fk : 0.f;
      F[e] = in ? F[e] : 1.f;
      E[e] = 1.f;
    }
  }

  // F: decays from the token's block's start up to it, E: behind it to the block's end
  f32x4_v A = {}, B = {};  // this wave's part; row 4 g + r, column m
  auto level = [&](auto half) {
    constexpr int H = decltype(half)::value;
    f32x4_v kk[4] = {}, qk[4] = {};  // short sums
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float from = k[e] * E[e];
      kk[e & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[e] * F[e], from, kk[e & 3], 0, 0, 0);
      qk[e & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[e] * F[e], from, qk[e & 3], 0, 0, 0);
    }
    kk[0] = kk[0] + kk[1] + (kk[2] + kk[3]);
    qk[0] = qk[0] + qk[1] + (qk[2] + qk[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g + r;
      const bool pair = ((i ^ m) & -H) == H && (i & H);
      A[r] = pair ? kk[0][r] : A[r];
      B[r] = pair ? qk[0][r] : B[r];
    }
    const bool upper = m & H;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float other = across<H>(F[e], upper);
      F[e] = upper ? F[e] * other : F[e];
      E[e] = upper ? E[e] : E[e] * other;
    }
  };
  level(std::integral_constant<int, 1>());
  level(std::integral_constant<int, 2>());
  level(std::integral_constant<int, 4>());
  level(std::integral_constant<int, 8>());
  sums[wid][0][lane] = A;
  sums[wid][1][lane] = B;

  // P k and P q as they are, P_15 / P k with token and channel exchanged
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    f32x4_v pk, pq, to;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      pk[r] = k[4 * s + r] * F[4 * s + r];
      pq[r] = q[4 * s + r] * F[4 * s + r];
      to[r] = k[4 * s + r] * E[4 * s + r];
    }
    ((f32x4_v*)ws)[(2 * wid + s) * 64 + 16 * g + place(m)] = pk;
    ((f32x4_v*)(ws + FRAG))[(2 * wid + s) * 64 + 16 * g + place(m)] = pq;
    *(f32x4_v*)&turn[wid][m][16 * s + 4 * g] = to;
    if (m == 15) {
      f32x4_v all;
#pragma unroll
      for (int r = 0; r < 4; ++r) all[r] = F[4 * s + r];
      ((f32x4_v*)(ws + AT_DECAY))[(2 * wid + s) * 4 + g] = all;
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    f32x4_v to;
#pragma unroll
    for (int r = 0; r < 4; ++r) to[r] = turn[wid][4 * r + g][16 * s + m];
    ((f32x4_v*)(ws + 2 * FRAG))[(2 * wid + s) * 64 + lane] = to;
  }
  if (wid == 1) {
    B = sums[0][1][lane] + sums[1][1][lane] + (sums[2][1][lane] + sums[3][1][lane]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ws[AT_B + 16 * place(4 * g + r) + place(m)] = 4 * g + r == m ? kq : B[r];
  }
  if (wid == 0) {
    A = sums[0][0][lane] + sums[1][0][lane] + (sums[2][0][lane] + sums[3][0][lane]);
    // lane m: column m of M; each row, once it is whole, is taken from all below it
    double M[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) M[i] = i == m ? 1. : 0.;
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      M[l] *= __int_as_float(__builtin_amdgcn_readlane(__float_as_int(beta), l));
#pragma unroll
      for (int i = l + 1; i < 16; ++i)
        M[i] -= M[l] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(A[i & 3]), 16 * (i >> 2) + l));
    }
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) ws[AT_M + 16 * place(i) + place(m)] = (float)M[i];
    }
  }
#endif
}

// grid (H, V / 16 CB, seqs), 8 + 2 CB waves.  Heads come first, so that the workgroups that read the
// same operands are on one XCD.
template <int CB>
__global__ __launch_bounds__(512 + 128 * CB, CB == 2 ? 6 : 5) void delta_chunk_scan_kernel(
    const DeltaArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  __shared__ f32x4_v parts[2][CB][8][64];  // of (P k)^T S0 and (P q)^T S0
  __shared__ f32x4_v us[CB][64];
  const int h = blockIdx.x, col0 = blockIdx.y * 16 * CB, seq = longest_first(a, blockIdx.z);
  const int ctx = a.ctx_lens[seq], len = a.seq_lens[seq] - ctx, chunks = (len + 15) / 16;
  const int64_t row0 = a.row_starts[seq], slot = a.slots[seq];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4;
  // The operands of a chunk, from a pointer that all lanes share and that stays at the last chunk
  const char* ahead =
      (const char*)(a.chunks + ((int64_t)h * (a.N / 16 + a.seqs) + row0 / 16 + seq) *
                                   DELTA_CHUNK_FLOATS);
  auto go_on = [&](int chunk) {  // from it to the next one
    ahead += chunk + 1 < chunks ? DELTA_CHUNK_FLOATS * 4 : 0;
  };
  auto operand = [&](unsigned at) { return *(const f32x4_v*)(ahead + at); };
  auto barrier = [&]() {  // of LDS alone: loads and stores stay under way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto sum = [&](int of, int c) {
    f32x4_v t[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = parts[of][c][i][lane];
    return (t[0] + t[1] + (t[2] + t[3])) + (t[4] + t[5] + (t[6] + t[7]));
  };
  // Two chunks a turn, whose operands are asked for two chunks ahead.  The loads ahead of the first
  // turn are in the order of a turn's, as otherwise every turn would wait for more than it needs
  auto turns = [&](auto&& step) {
    int chunk = 0;
    for (; chunk + 1 < chunks; chunk += 2) {
      step(std::integral_constant<int, 0>(), chunk);
      step(std::integral_constant<int, 1>(), chunk + 1);
    }
    if (chunk < chunks) step(std::integral_constant<int, 0>(), chunk);
  };

  if (wid < 8) {
    float* const state = a.state + (slot * a.H + h) * 128 * a.V + col0 + m;
    f32x4_v S[CB], pk[2], pq[2], to[2], decay[2];
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[c][r] = ctx > 0 ? state[(int64_t)channel_of(wid, g, r) * a.V + 16 * c] : 0.f;
    const unsigned at = (wid * 64 + lane) * 16, at_decay = (AT_DECAY + (wid * 4 + g) * 4) * 4;
    auto ask = [&](f32x4_v& x, unsigned from) {
      x = operand(from);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ask(pk[i], at);
      ask(pq[i], at + FRAG * 4);
      ask(decay[i], at_decay);
      ask(to[i], at + FRAG * 8);
      go_on(i);
    }
    // products by an operand, the columns' side by side, since each waits for its last one
    auto products = [&](f32x4_v* y, f32x4_v x, const f32x4_v* by) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < CB; ++c)
          y[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r], by[c][r], y[c], 0, 0, 0);
    };
    turns([&](auto fixed, int chunk) {
      constexpr int i = decltype(fixed)::value;
      f32x4_v y[CB] = {}, z[CB] = {}, u[CB];
      products(y, pk[i], S);
#pragma unroll
      for (int c = 0; c < CB; ++c) parts[0][c][wid][lane] = y[c];
      ask(pk[i], at);
      barrier();
      products(z, pq[i], S);  // while u is made
#pragma unroll
      for (int c = 0; c < CB; ++c) parts[1][c][wid][lane] = z[c];
      ask(pq[i], at + FRAG * 4);
#pragma unroll
      for (int c = 0; c < CB; ++c) S[c] *= decay[i];
      ask(decay[i], at_decay);
      barrier();
#pragma unroll
      for (int c = 0; c < CB; ++c) u[c] = us[c][lane];
      products(S, to[i], u);
      ask(to[i], at + FRAG * 8);
      go_on(chunk + 2);
    });
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        state[(int64_t)channel_of(wid, g, r) * a.V + 16 * c] = S[c][r];
  } else if (wid < 8 + CB) {
    const int mine = wid - 8;
    const unsigned at = (AT_M + (m * 4 + g) * 4) * 4, row = a.C * sizeof(bf16_t);
    const char* values = (const char*)((const bf16_t*)a.y + row0 * a.C + 2 * a.G * 128 + h * a.V +
                                       col0 + 16 * mine);
    f32x4_v M[2];
    bf16_t v[2][4];
    auto fetch = [&](int i, int chunk) {  // of tokens past the end the last one's
      M[i] = operand(at);
      __builtin_amdgcn_sched_barrier(0);
      const unsigned most = len - 1 - 16 * min(chunk, chunks - 1);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v[i][r] = *(const bf16_t*)(values + __umul24(min(4u * r + g, most), row) + m * sizeof(bf16_t));
      __builtin_amdgcn_sched_barrier(0);
      values += chunk + 1 < chunks ? 16 * row : 0;
      go_on(chunk);
    };
    fetch(0, 0);
    fetch(1, 1);
    __builtin_amdgcn_s_setprio(3);  // all others wait for it
    turns([&](auto fixed, int chunk) {
      constexpr int i = decltype(fixed)::value;
      barrier();
      f32x4_v x = sum(0, mine);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = to_f(v[i][r]) - x[r];
      us[mine][lane] = causal(M[i], x, f32x4_v{});
      barrier();
      fetch(i, chunk + 2);
    });
  } else {
    const int mine = wid - 8 - CB;
    const unsigned at = (AT_B + (m * 4 + g) * 4) * 4;
    f32x4_v B[2];
    for (int i = 0; i < 2; ++i) {
      B[i] = operand(at);
      go_on(i);
    }
    float* const out = a.o + (row0 * a.H + h) * a.V + col0 + 16 * mine + m;
    turns([&](auto fixed, int chunk) {
      constexpr int i = decltype(fixed)::value;
      barrier();
      barrier();
      const f32x4_v o = causal(B[i], us[mine][lane], sum(1, mine));
      B[i] = operand(at);
      go_on(chunk + 2);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * chunk + 4 * r + g;
        if (t < len) out[(int64_t)t * a.H * a.V] = o[r];
      }
    });
  }
  if (blockIdx.y == 0) keep_inputs<bf16_t>(a, h, ctx, len, row0, slot);
#endif
}

// columns: 16s of columns a workgroup, 1 or 2
extern "C" void launch_delta_chunks(const DeltaArgs* args, int columns, hipStream_t stream) {
  const DeltaArgs a = *args;
  delta_chunk_kernel<<<dim3(a.n_tiles, a.H), 256, 0, stream>>>(a);
  if (columns == 2)
    delta_chunk_scan_kernel<2><<<dim3(a.H, a.V / 32, a.seqs), 768, 0, stream>>>(a);
  else
    delta_chunk_scan_kernel<1><<<dim3(a.H, a.V / 16, a.seqs), 640, 0, stream>>>(a);
}
