"""Op dispatch.

Two implementations of every engine op:

- ``reference`` — plain PyTorch fp32, runs on CPU.  The numerics oracle for
  every HIP kernel test and the compute path for CPU-only engine tests.
- ``hip`` — hand-written CDNA4 HIP kernels (csrc/*.hip) through the in-tree
  ``_C`` extension.  The ONLY path on a GPU: if a tensor is on cuda and the
  extension is missing, ops raise instead of silently falling back, so a GPU
  run that passes is guaranteed to have run the native kernels.
"""
from __future__ import annotations

from typing import NamedTuple, Optional

import torch

_HIP = None
_HIP_ERR: Exception | None = None


def _hip():
    global _HIP, _HIP_ERR
    if _HIP is None and _HIP_ERR is None:
        try:
            from . import hip as m

            _HIP = m
        except Exception as e:  # pragma: no cover
            _HIP_ERR = e
    if _HIP is None:
        raise RuntimeError(
            f"HIP ops extension not available on a GPU tensor path: {_HIP_ERR}\n"
            "Build it with: python build_ext.py (PYTORCH_ROCM_ARCH=gfx950)"
        )
    return _HIP


def _impl(t: torch.Tensor):
    if t.is_cuda:
        return _hip()
    from . import reference as m

    return m


import os

# Rows from which linear() takes csrc/linear.hip whatever the sizes; step_linear() has a rule
_GEMM_MIN_M = int(os.environ.get("ACP_GEMM_MIN_M", str(1 << 30)))


def linear(x, w, bias=None):
    """x[*, K] @ w[N, K]^T (+ bias[N]) → [*, N] by the library, unless ACP_GEMM_MIN_M says
    otherwise for that many bf16 rows."""
    if (
        x.is_cuda
        and bias is None
        and x.dtype == torch.bfloat16
        and x.dim() == 2
        and x.shape[0] >= _GEMM_MIN_M
        and w.shape[0] % 256 == 0
        and w.shape[1] % 128 == 0
    ):
        return _hip().gemm_bf16(x, w)
    return torch.nn.functional.linear(x, w, bias)


def _few_rows_pay(m: int, outs: int, k: int, glu: bool) -> bool:
    """Whether csrc/step_linear.hip is the faster one for m rows, outs outputs (of a GLU: pairs)
    and k inner elements; the GEMM library (with a pass of its own for the GLU) is in brackets, us
    of every weight from memory.  Up to 4096 elements at nearly all sizes: one row 4096 x 4096 8.1
    (15), 20048 x 2048 16 (49), four rows 6144 x 4096 13.6 (15.1), pairs of 14336 x 4096 41 (64), but
    short rows of many outputs not, 65536 x 1024 30 (27).  Above that not
    where few outputs are long sums, 512 x 14336 17 (13), 16 x 5120 9 (7.5), pairs of 2048 x 7168 19.5
    (17.1), nor between one and two workgroups a CU, four rows 4608 x 4608 13.7 (12.2), 6144 x 7168
    20.3 (19.1), pairs of 5632 x 14336 68 (63), where the second round is not full; rows that are no
    multiples of 512 are the library's slow ones, four rows 6144 x 8064 22 (29), pairs of 2048 x
    11008 23 (37)."""
    if m > 4:
        return False
    if k < 1536:
        return outs <= 28672
    if k <= 4096:
        return True
    if glu and k <= 5120:
        return outs >= 64
    if glu:
        return (
            (k <= 6144 or 8192 < k <= 11008) and outs >= 2048
            or 7680 < k < 8192 and (outs <= 64 or 512 <= outs)
            or outs >= 4096 and not (k > 11008 and 4096 < outs < 8192)
        )
    if 4096 < outs < 8192:
        return outs >= 6144 and (m == 1 or k % 512 > 0)
    if k <= 5120:
        return outs >= 64
    return outs >= 2048 or 7680 < k < 8192 and (outs <= 64 or 512 <= outs)


def _rows(t) -> bool:
    """Rows of 16-byte units."""
    return (
        t.dim() == 2
        and t.is_cuda
        and t.dtype == torch.bfloat16
        and t.stride(1) == 1
        and (t.shape[0] == 1 or t.stride(0) % 8 == 0)
        and t.data_ptr() % 16 == 0
    )


def _recorded(*ts) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in ts)


def _whole(t) -> bool:
    """No subclass, which may have a product of its own."""
    return type(t) in (torch.Tensor, torch.nn.Parameter)


def _followed() -> bool:
    """Whether something follows the library's calls, which kernels of our own are not seen by:
    transforms, forward-mode derivatives, dispatch modes, a trace, a compiler, autocast."""
    return (
        torch.compiler.is_compiling()
        or torch._C._functorch.peek_interpreter_stack() is not None
        or torch.autograd.forward_ad._current_level >= 0
        or torch._C._len_torch_dispatch_stack() > 0
        or torch._C._get_tracing_state() is not None
        or torch.is_autocast_enabled("cuda")
    )


def _few_rows(x, w, bias=None, glu: bool = False) -> bool:
    """Whether csrc/step_linear.hip takes x w^T: what it can, at the sizes at which it pays.
    It has no derivative: what autograd records or others follow is left to the library."""
    return (
        0 < x.shape[0] <= 4
        and _whole(x)
        and _whole(w)
        and not _followed()
        and _rows(x)
        and _rows(w)
        and x.device == w.device
        and x.shape[1] == w.shape[1]
        and w.shape[0] > 0
        and w.shape[1] > 0
        and w.shape[1] % 32 == 0
        and _few_rows_pay(x.shape[0], w.shape[0] >> glu, w.shape[1], glu)
        and (
            bias is None
            or _whole(bias) and bias.is_cuda and bias.dtype == torch.bfloat16
            and bias.is_contiguous() and bias.shape == w.shape[:1]
        )
        and not _recorded(x, w, bias)
    )


def _many_rows_pay(m: int, n: int, k: int, glu: bool, adds: bool = False) -> bool:
    """Whether csrc/linear.hip is the faster one for m rows, n outputs (of a GLU: gates and ups)
    and k inner elements, where ``adds``: what reads it adds up its parts, which saves a launch of
    4.3 us.  The GEMM library (with a pass of its own for the GLU) is in brackets, us of every
    weight from memory.  Up to about 2000 rows at most sizes: 8 x 22016 x 4096 GLU 33 (55), 64 x
    4096 x 14336 29 (43), 192 x 4096 x 4096 22 (34), 512 x 6288 x 2048 22 (26), 1739 x 4096 x 11008 130
    (159), 24 x 128256 x 4096 167 (195).  Without ``adds`` not: up to 32 rows of medium weights, 8 x
    6144 x 4096 17.2 (16.5), 32 x 7168 x 4096 22.4 (17.6), 16 x 4096 x 8192 19.6 (17.9), or few outputs, 8 x
    2048 x 8192 13.7 (12.4); where unsplit tiles leave half of the CUs idle and parts gain little, 80 x
    2048 x 4096 12.0 (11.3), 61 x 3584 x 3584 12.5 (11.0), 33 to 64 x 4096 x 4096 within 5% either way; weights
    that two tiles of rows read, 128 x 12288 x 4096 38 (35), 96 of them 34 (34).  The library has other
    sizes of its own beside slow ones, 61 x 6144 x 4096 20.6 (19.5), 160 x 12288 x 4096 40.2 (39.5): not told
    apart.  From 1024
    rows on (2048 with a GLU or ``adds``) it is 2 to 9% ahead where
    256 x 256 tiles fill their last round, 1400 x 32000 x 4096 301 (287), 5000 x 6144 x 4096 188 (179),
    7664 x 2048 x 8192 190 (174), 8131 x 4096 x 4096 195 (183), but not for the GLU, 7664 x 28672 x 4096 1287 (1380),
    for outputs that are no whole tiles, 7664 x 17744 x 2048 424 (506), and for rows that
    together are beyond the memory-side cache, 7664 x 4096 x 14336 619 (1001); with a last
    round that is not full it is slower, 5000 x 4096 x 4096 134 (141), 10000 x 4096 x 4096 243 (373)."""
    if m <= 4 or n * k < 1 << 21:
        return False
    plain = not (glu or adds)
    if plain and m <= 32:
        medium = 4096 <= k <= 8192 and n <= 8192 and n * k >= 24 << 20
        return not (medium or (m <= 16 and k >= 4 * n))
    if plain and 3584 <= k < 8192 and -(-m // 32) * n <= 8192:
        return False
    if plain and k >= 4096 and 64 < m <= 128 and 10240 < n < 16384:
        return False
    if m < (1024 if plain else 2048) or glu or n % 256 or m * k >= 100 << 20:
        return True
    tiles = -(-m // 256) * (n // 256)
    return tiles < 0.93 * 256 * -(-tiles // 256)


def _many_rows(x, w, bias=None, glu: bool = False, out=None, adds: bool = False) -> bool:
    """Whether csrc/linear.hip takes x w^T: what it can, at the sizes at which it pays.  It has
    no derivative and is not seen by what follows the library's calls: that is left to it."""

    def below_2gib(t):
        return (t.shape[0] - 1) * t.stride(0) + t.shape[1] < 1 << 30

    return (
        x.dim() == 2
        and w.dim() == 2
        and x.shape[1] == w.shape[1]
        and w.shape[1] % 64 == 0
        and w.shape[0] % (16 if glu else 8) == 0
        and _many_rows_pay(x.shape[0], w.shape[0], w.shape[1], glu, adds)
        and _whole(x)
        and _whole(w)
        and not _followed()
        and _rows(x)
        and _rows(w)
        and x.device == w.device
        and below_2gib(x)
        and below_2gib(w)
        and (out is None or _rows(out))
        and (
            bias is None
            or _whole(bias) and bias.device == x.device and bias.dtype == torch.bfloat16
            and bias.is_contiguous() and bias.shape == w.shape[:1] and bias.data_ptr() % 16 == 0
        )
        and not _recorded(x, w, bias)
    )


def step_linear(x, w, bias=None):
    """linear() of a step's activations in a model's forward pass: rows of 16 bits go to kernels of
    their own where those are the faster ones, unless autograd records them."""
    if _few_rows(x, w, bias):
        return _hip().step_linear(x, w, bias)
    if _many_rows(x, w, bias):
        return _hip().linear(x, w, bias)
    return linear(x, w, bias)


def step_linear_swiglu(x, w):
    """swiglu(step_linear(x, w)), in one pass where step_linear() has a kernel of its own."""
    if w.shape[0] % 16 == 0 and _few_rows(x, w, None, True):
        return _hip().step_linear(x, w, None, True)
    if _many_rows(x, w, None, True):
        return _hip().linear(x, w, unit="swiglu")
    return swiglu(linear(x, w))


def step_linear_glu(x, w, glu, out):
    """clamped_glu(step_linear(x, w)) -> out [N, I] (row-strided), likewise.  ``glu`` has limit,
    alpha, offset and maybe cubic."""
    cubic = getattr(glu, "cubic", 0.0)
    if _many_rows(x, w, None, True, out):
        _hip().linear(x, w, None, "glu", (glu.limit, glu.alpha, glu.offset, cubic), out)
    else:
        clamped_glu(step_linear(x, w), glu.limit, glu.alpha, glu.offset, out, cubic)


def step_linear_add_rmsnorm(x, w, residual, weight, eps: float = 1e-5):
    """fused_add_rmsnorm(step_linear(x, w), residual, weight, eps); a product in parts leaves
    their sum to the norm's pass."""
    if (
        _many_rows(x, w, adds=True)
        and w.shape[0] <= _hip()._C.ADD_RMSNORM_MOST
        and all(
            t.dtype == x.dtype and t.device == x.device and t.is_contiguous()
            and t.data_ptr() % 16 == 0 for t in (residual, weight)
        )
        and residual.shape == (x.shape[0], w.shape[0])
        and weight.shape == w.shape[:1]
    ):
        return _hip().linear_add_rmsnorm(x, w, residual, weight, eps)
    return fused_add_rmsnorm(step_linear(x, w), residual, weight, eps)


def step_linear_rope_and_cache(x, w, heads: int, positions, slot_mapping, k_cache, v_cache,
                               cos_sin):
    """rope_and_cache() of step_linear(x, w), rows of ``heads`` queries, then keys, then values as
    the caches [.., Hkv, D] hold them, with a product in parts added up in its pass.  Returns the
    queries [N, heads, D]."""
    kv, d = k_cache.shape[-2:]
    caches = (positions, slot_mapping, k_cache, v_cache, cos_sin)
    if (
        _many_rows(x, w, adds=True)
        and d % 128 == 0
        and w.shape[0] == (heads + 2 * kv) * d
        and k_cache.shape == v_cache.shape
        and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in caches[2:])
        and k_cache.dtype == v_cache.dtype == x.dtype
        and positions.numel() == slot_mapping.numel() == x.shape[0]
    ):
        return _hip().linear_rope_and_cache(x, w, heads, *caches)
    y = step_linear(x, w)
    y = y.view(-1, heads + 2 * kv, d)
    return rope_and_cache(y[:, :heads], y[:, heads:-kv], y[:, -kv:], *caches)[0]


def linear_add_(y, x, w):
    """y += x @ w^T in one GEMM."""
    return y.addmm_(x, w.t())


def rmsnorm(x, weight, eps: float = 1e-5):
    return _impl(x).rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x, residual, weight, eps: float = 1e-5):
    """returns (normed, new_residual) where new_residual = x + residual."""
    return _impl(x).fused_add_rmsnorm(x, residual, weight, eps)


def rope_and_cache(q, k, v, positions, slot_mapping, k_cache, v_cache, cos_sin):
    """Apply rotary embedding to q,k in place and scatter k,v into the paged
    cache at slot_mapping.  q:[N, Hq, D] k/v:[N, Hkv, D]."""
    return _impl(q).rope_and_cache(q, k, v, positions, slot_mapping, k_cache, v_cache, cos_sin)


def attention_prefill(q, k_cache, v_cache, block_table, seq_len, ctx_len, scale):
    """Causal attention for ONE sequence's prefill chunk (test/oracle entry).
    q: [Lq, Hq, D]; KV read from the paged cache; ctx_len = tokens already
    cached before this chunk (the chunk's causal offset)."""
    return _impl(q).attention_prefill(q, k_cache, v_cache, block_table, seq_len, ctx_len, scale)


def attention_prefill_batch(q, k_cache, v_cache, batch, scale, out=None):
    """Causal attention for ALL prefill chunks of a FlatBatch in one launch.
    q: [num_prefill_tokens, Hq, D]."""
    return _impl(q).attention_prefill_batch(q, k_cache, v_cache, batch, scale, out)


def attention_decode_batch(q, k_cache, v_cache, batch, scale, out=None):
    """One-token-per-sequence paged attention.  q: [B, Hq, D]."""
    return _impl(q).attention_decode_batch(q, k_cache, v_cache, batch, scale, out)


def swiglu(gate_up):
    """gate_up: [N, 2*I] (gate | up interleaved as two halves) → [N, I]."""
    return _impl(gate_up).swiglu(gate_up)


# ------------------------------------------------ fp32-residual norms, GLU, gates


def layernorm(x, weight, eps: float, dtype):
    """Layer norm without bias of an fp32 residual [N, K] -> dtype."""
    return _impl(x).layernorm(x, weight, eps, dtype)


class Depth(NamedTuple):
    """States of a depth average: X_0 (the embedding output) and every layer's result."""

    states: torch.Tensor   # [layers + 1, N, K] fp32
    coef: torch.Tensor     # [layers, layers + 1] fp32: row i weighs the states after layer i
    partial: torch.Tensor  # [DEPTH_AHEAD, N, K] fp32 workspace

    @staticmethod
    def new(coef: torch.Tensor, N: int, K: int) -> "Depth":
        planes = torch.empty(
            coef.shape[1] + DEPTH_AHEAD, N, K, dtype=torch.float32, device=coef.device
        )
        return Depth(planes[: coef.shape[1]], coef, planes[coef.shape[1] :])


#: sums the first layer of a block prepares for the block's others (csrc/residual_norm.h)
DEPTH_AHEAD = 3


def residual_norm(x, y, eps: float, y_norm=None, x_norm=None, out=None, *, center=True,
                  offset: float = 0.0, mult: float = 1.0, depth: Optional[Depth] = None,
                  layer: int = 0, x_norm2=None, out2=None, experts=None, gate=None):
    """x += mult * y, or x += mult * rmsnorm(y) * y_norm, in the fp32 residual x, where
    ``experts`` (rows [N, k, K], weights [N, k] fp32) joins y as
    sum_j weights[:, j] * rows[:, j] and then ``gate`` [N, K] (row-strided) multiplies it
    by its sigmoid; then, with ``depth``, x is filed as layer ``layer``'s state and replaced by
    sum_j coef[layer, j] * states[j] (layers in order: later ones use sums made by
    earlier ones); then out = norm(x) * x_norm, or x itself without x_norm.  The norm
    of x is a layer norm, an RMS norm if not ``center``; ``offset`` is added to the
    norm weights.  out2 is the same norm under the weight x_norm2."""
    return _impl(x).residual_norm(
        x, y, eps, y_norm, x_norm, out, center, offset, mult, depth, layer, x_norm2, out2,
        experts, gate,
    )


def embed_positions(token_ids, positions, table, cos_sin, x, copy=None, scale: float = 1.0):
    """x = copy = scale * table[token] plus, with cos_sin [2, P, ceil(K / 2)], sin (even
    entries) and cos (odd entries) of the position's angles; x, copy fp32 [N, K]."""
    return _impl(x).embed_positions(token_ids, positions, table, cos_sin, x, copy, scale)


def softcap(logits, cap):
    """cap * tanh(logits / cap) in fp32; the logits in fp32 without a cap."""
    return logits.float() if cap is None else _impl(logits).softcap(logits, cap)


def clamped_glu(gate_up, limit: float, alpha: float, offset: float, out, cubic: float = 0.0):
    """gate_up [N, 2I] (row-strided halves) -> out [N, I] (row-strided):
    g * sigmoid(alpha (g + cubic g^3)) * (u + offset), g capped at limit, u at +-limit."""
    return _impl(gate_up).clamped_glu(gate_up, limit, alpha, offset, out, cubic)


def step_linear_parts(x, w):
    """step_linear(x, w), or the parts of it [parts, N, O] in fp32, which what reads them adds up in their
    order."""
    if _many_rows(x, w, adds=True):
        return _hip()._C.linear_parts(x, w)
    return step_linear(x, w)


def side_layer_fits(x, gate, *weights) -> bool:
    """Whether side_layer() takes this residual, this side gate and these other weights.  Its product is
    the library's, as of linear(), where autograd records it or others follow it."""
    return (
        x.is_cuda
        and all(map(_whole, (x, gate, *weights)))
        and not _followed()
        and not _recorded(x, gate, *weights)
        and _hip().side_layer_fits(x, gate, *weights)
    )


def side_layer(x, y, gate, token_ids, table, offset: int, proj, eps: float, y_norm, x_norm, out):
    """side_gate(x, y, ...), its product with proj, and residual_norm() of that, in one launch: x is updated
    in place, out as of residual_norm().  y may be a product's parts (step_linear_parts())."""
    _hip().side_layer(x, y, gate, token_ids, table, offset, proj, eps, y_norm, x_norm, out)


def side_gate(x, y, gate, token_ids, table, offset: int):
    """The fp32 residual x + y (x itself may be reused for it) and
    gelu_tanh(gate (x + y)) * table[token, offset : offset + D]: [N, D]."""
    return _impl(x).side_gate(x, y, gate, token_ids, table, offset)


# ------------------------------------------------------------ latent attention

#: latent sizes the MFMA kernels are built for; larger ones run the plain kernel
LATENT_RANKS = (64, 128, 256, 384, 512)


def latent_rank(kv_rank: int) -> int:
    """The padded latent size kernels and caches use for kv_rank."""
    for r in LATENT_RANKS:
        if kv_rank <= r:
            return r
    return -(-kv_rank // 64) * 64


#: query/key and value head sizes of the expanded prefill kernel
LATENT_HEADS = (64, 128, 256)


def latent_head(dim: int) -> int:
    """The padded per-head size for dim."""
    for n in LATENT_HEADS:
        if dim <= n:
            return n
    return -(-dim // 64) * 64


def latent_inputs(kv, norm_w, eps: float, kv_rank: int, rot_dim: int, rank: int,
                  positions, slot_mapping, cos_sin, cache, q=None, q_norm=None, q_rank=0, glu=None):
    """kv [N, kv_rank + rot_dim] (row-strided): RMS-norm the latent, rotate the
    key part (interleaved pairs), scatter [latent -> rank | rotated] rows into
    cache [blocks, block, row].  With q [N, K] (low-rank query, row-strided; its
    columns past q_rank are zero padding) returns rmsnorm(q) * q_norm.  With glu (out, gate_up, limit,
    alpha, offset) does that clamped_glu() of as many rows as well."""
    return _impl(kv).latent_inputs(
        kv, norm_w, eps, kv_rank, rot_dim, rank, positions, slot_mapping, cos_sin, cache,
        q, q_norm, q_rank, glu,
    )


def head_linear(x, w, out, gate=None):
    """out[n, h] = w[h] @ x[n, h], times sigmoid(gate[n, h]) if given.
    x [N, H, K], w [H, O, K], out [N, H, O]; x, out, gate row-strided."""
    return _impl(x).head_linear(x, w, out, gate)


def latent_attention(q, q_rot, cos_sin, rot_dim: int, cache, batch, scale: float, window,
                     row0: int = 0, skip=(), sink=None):
    """Softmax attention of absorbed queries over cached rows (``sink`` [H], fp32, or None
    joins the denominator), for a FlatBatch's token rows row0.. except the prefill chunks in ``skip`` (left undefined).
    q [N, H, rank] and its part q_rot [N, H, rot] still to be rotated by the
    row's position; values are a cache row's first ``rank`` dims.
    window = visible keys per query, None = all.  Returns [N, H, rank]."""
    return _impl(q).latent_attention(
        q, q_rot, cos_sin, rot_dim, cache, batch, scale, window, row0, skip, sink
    )


def latent_values(q, q_rot, cos_sin, rot_dim: int, cache, batch, scale: float, window,
                  row0: int, skip, sink, w, out, gate=None):
    """head_linear(latent_attention(...), w, out, gate)."""
    if q.is_cuda:
        return _hip().latent_values(
            q, q_rot, cos_sin, rot_dim, cache, batch, scale, window, row0, skip, sink, w, out, gate
        )
    latent = latent_attention(
        q, q_rot, cos_sin, rot_dim, cache, batch, scale, window, row0, skip, sink
    )
    return head_linear(latent, w, out, gate)


def can_expand(t, d: int, v: int, rot: int) -> bool:
    """Is there a kernel for expanded keys and values of these padded sizes?"""
    return t.is_cuda and _hip().can_expand(t.dtype, d, v, rot)


def latent_expanded_prefill(q, w_ukv, gate, cos_sin, rot_dim: int, cache, batch, chunks,
                            rank: int, scale: float, window, out, sink=None):
    """The prefill chunks ``chunks`` with keys and values expanded from their
    cached latents by w_ukv [H*d + H*v, rank]; q [N, H, d + rot] not rotated.
    Writes the chunks' rows of out [N, H, v], gated."""
    _hip().latent_expanded_prefill(
        q, w_ukv, gate, cos_sin, rot_dim, cache, batch, chunks, rank, scale, window, out, sink
    )


# ---------------------------------------- grouped attention: caps, windows, sinks


def cache_keys_values(k, v, slot_mapping, k_cache, v_cache):
    """Scatter k [N, G, d], v [N, G, e] (row-strided) into paged caches
    [blocks, block, G, d or e]."""
    return _impl(k).cache_keys_values(k, v, slot_mapping, k_cache, v_cache)


def attention_inputs(proj, heads: int, dim: int, vdim: int, k_cache, v_cache, batch, eps: float,
                     *, conv=None, ring=None, q_norm=None, k_norm=None, v_norm: bool = False,
                     cos_sin=None, head_mult=None, q_temp=None):
    """From projected rows [N, q | k | v channels] (row-strided; heads padded from dim and
    vdim to the caches' d and e) to queries [N, heads, d], which are returned, and keys
    and values in their cache slots (batch.slot_mapping).  In this order, each optional:

    conv [taps, channels]: causal convolution per channel; the last inputs of a
        sequence are kept by position in its slot of ``ring`` [slots, taps, channels]
    q_norm, k_norm [d], v_norm: RMS norm per head over dim or vdim; [heads * d] and
        [G * d]: over all heads at once (no conv, no v_norm)
    cos_sin [2, P, n]: rotate a query's and key's first n pairs (2i, 2i + 1)
    head_mult [heads] fp32, q_temp (coef, every): queries times the head's factor, and
        times 1 + coef ln(floor((p + 1) / every) + 1) at position p"""
    return _impl(proj).attention_inputs(
        proj, heads, dim, vdim, k_cache, v_cache, batch, eps, conv, ring, q_norm, k_norm,
        v_norm, cos_sin, head_mult, q_temp,
    )


def grouped_attention(q, k_cache, v_cache, batch, scale: float, cap, window, keep_first: int,
                      sink, out, bias=None, sigmoid: bool = False, gate=None, chunk=None,
                      talk=None):
    """Attention of a FlatBatch's rows over the paged cache; query head n uses
    key/value head n // (H / G).  ``talk`` [H, H] (fp32, of values that the
    model's dtype holds) mixes the scores over the heads: head h's are
    sum_g talk[h, g] * head g's.  Scores are capped if ``cap``; a query sees
    itself and the ``window`` - 1 tokens before it (None = all) and the ``keep_first``
    first tokens, with ``chunk`` (no keep_first) only those of its own chunk, position
    // chunk; ``sink`` [H] (fp32) or None joins the softmax denominator.
    ``bias`` [H, D] (fp32) adds bias[h, min(distance, D - 1)] to the capped scores;
    ``sigmoid``: weights are the scores' sigmoids, not a softmax; ``gate`` [N, H]
    (row-strided) multiplies a head's output by its sigmoid.
    q [N, H, d], out [N, H, e], both row-strided."""
    return _impl(q).grouped_attention(
        q, k_cache, v_cache, batch, scale, cap, window, keep_first, sink, out, bias, sigmoid,
        gate, chunk, talk,
    )


# -------------------------------------------------------------------- experts


def moe_route(h, router, bias, top: int, sigmoid: bool = False, scale: float = 1.0):
    """The ``top`` experts with the largest logits router @ h + bias (fp32) of every row:
    ids [N, top] int32 and scale * the softmax over the chosen logits [N, top] fp32.
    ``sigmoid``: the choice is by sigmoid(router @ h) + bias, the weights are
    scale * the chosen sigmoids over their sum."""
    return _impl(h).moe_route(h, router, bias, top, sigmoid, scale)


def moe_experts(h, gate_up, down, ids, glu):
    """Every chosen expert's GLU of its row: h [N, K], gate_up [E, 2I, K], down [E, W, I],
    ids [N, k] -> [N, k, W].  ``glu`` has limit, alpha, offset and cubic."""
    return _impl(h).moe_experts(h, gate_up, down, ids, glu)


# ----------------------------------------------------------------- delta rule


def gated_delta_bytes(tokens: int, H: int, D: int, V: int, dtype) -> int:
    """What gated_delta() holds on the GPU for a step of so many prompt tokens, beyond what grows with a layer's
    activations."""
    return _hip().gated_delta_bytes(tokens, H, D, V, dtype)


def gated_delta(qkv, conv, b, z, A_log, dt_bias, gate, norm, eps: float, unit_eps: float,
                kv_heads: int, state, conv_state, batch, gate_silu: bool = False):
    """Gated delta rule over a FlatBatch's rows, each sequence from the state in its
    slot (zero at position 0), which is advanced.  Row-strided inputs: qkv
    [N, 2*G*D + H*V] before the convolution, b [N, H] before its sigmoid, z [N, H*D]
    or [N, H] (one decay per head) the decays' input, gate [N, H*V] before its sigmoid or
    silu.  conv [channels, taps]; fp32: A_log [H], dt_bias like z, norm [V], state
    [slots, H, D, V]; conv_state [slots, taps, channels], the last convolution inputs in a
    ring by position.  Returns [N, H*V]: normed per head and gated."""
    return _impl(qkv).gated_delta(
        qkv, conv, b, z, A_log, dt_bias, gate, norm, eps, unit_eps, kv_heads, state,
        conv_state, batch, gate_silu,
    )


def softmax_sample(logits, temperatures, top_ks, top_ps, gen, mask=None,
                   uniforms=None, mask_map=None):
    """Batch sampling: temperature/top-k/top-p with optional boolean vocab
    masks (constrained decoding; compact [M, V] rows + mask_map [B]
    indirection for BPE-scale vocabularies) and optional precomputed
    per-row uniforms (per-request seeded generators).  Returns [B] long."""
    return _impl(logits).softmax_sample(
        logits, temperatures, top_ks, top_ps, gen, mask, uniforms, mask_map
    )
