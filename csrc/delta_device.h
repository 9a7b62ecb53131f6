// What the kernels of the gated delta rule share (device code).
#pragma once
#include "common_t.h"
#include "gated_delta.h"

// log(1 + e^x) with a small relative error everywhere: log(u) e / (u - 1), u = 1 + e
DEV float softplus_f(float x) {
  if (x > 20.f) return x;
  const float e = __expf(x), u = 1.f + e;
  return u == 1.f ? e : __logf(u) * e * __builtin_amdgcn_rcpf(u - 1.f);
}

// rate = exp(A_log)
DEV float decay_f(float z, float rate) { return __expf(-rate * softplus_f(z)); }

// The sequence of workgroups z.  The longest ones come first, as workgroups start in order of
// z and a sequence's tokens are a serial chain, and they go first on a SIMD, too: 16 heads of 128,
// 5 sequences of 571 to 2536 tokens, token by token, 687 us as they came, 556 longest first; 12 of 443
// to 2536 979, 920 in order, 884 with priorities.  More than a wave's lanes: as they come.
static DEV int longest_first(const DeltaArgs& a, int z) {
  if (a.seqs == 1 || a.seqs > 64) return z;
  const int lane = threadIdx.x & 63, at = min(lane, a.seqs - 1);
  const int len = a.seq_lens[at] - a.ctx_lens[at];
  int rank = 0, most = 0;
  for (int i = 0; i < a.seqs; ++i) {
    const int other = __builtin_amdgcn_readlane(len, i);
    rank += other > len || (other == len && i < lane);
    most = max(most, other);
  }
  const int seq = __builtin_ctzll(__ballot(lane < a.seqs && rank == z));
  const int mine = __builtin_amdgcn_readlane(len, seq);
  if (mine > most / 4 * 3) __builtin_amdgcn_s_setprio(3);
  else if (mine > most / 2) __builtin_amdgcn_s_setprio(2);
  else if (mine > most / 4) __builtin_amdgcn_s_setprio(1);
  return seq;
}

// The last convolution inputs of head h's channels into the ring, once the old ones have been read
template <typename T>
DEV void keep_inputs(const DeltaArgs& a, int h, int ctx, int len, int64_t row0, int64_t slot) {
  const int group = a.H / a.G, kvh = h / group;
  const int total = (h % group == 0 ? 2 * a.D : 0) + a.V;
  T* ring = (T*)a.ring + slot * a.taps * a.C;
  for (int i = threadIdx.x; i < total; i += blockDim.x) {
    const int c = i < a.V ? 2 * a.G * a.D + h * a.V + i
                : i < a.V + a.D ? kvh * a.D + i - a.V : (a.G + kvh) * a.D + i - a.V - a.D;
    for (int t = max(0, len - a.taps); t < len; ++t)
      ring[(int64_t)((ctx + t) % a.taps) * a.C + c] =
          ((const T*)a.qkv)[(row0 + t) * a.qkv_stride + c];
  }
}
