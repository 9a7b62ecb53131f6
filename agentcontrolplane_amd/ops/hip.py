"""GPU op dispatch into the hand-written CDNA4 kernels (csrc/*.hip).

No fallbacks: a cuda-tensor call that cannot reach a kernel raises, so a
passing GPU run proves the native path ran (the round-end loader check
looks for agentcontrolplane_amd/_C.so in the process maps).
"""
from __future__ import annotations

import torch

from .. import _C  # in-tree extension; ImportError surfaces via ops.__init__


def rmsnorm(x, weight, eps: float = 1e-5):
    out = torch.empty_like(x)
    _C.rmsnorm(out, x, weight, eps)
    return out


def fused_add_rmsnorm(x, residual, weight, eps: float = 1e-5):
    out = torch.empty_like(x)
    _C.fused_add_rmsnorm(out, residual, x, weight, eps)  # residual updated in place
    return out, residual


def linear_add_rmsnorm(x, w, residual, weight, eps: float):
    y = _C.linear_parts(x, w)
    if y.dim() == 2:
        return fused_add_rmsnorm(y, residual, weight, eps)
    out = torch.empty_like(residual)
    _C.parts_add_rmsnorm(out, residual, y, weight, eps)
    return out, residual


def linear_rope_and_cache(x, w, heads: int, positions, slot_mapping, k_cache, v_cache, cos_sin):
    y = _C.linear_parts(x, w)
    kv, d = k_cache.shape[-2:]
    if y.dim() == 2:
        y = y.view(-1, heads + 2 * kv, d)
        return rope_and_cache(
            y[:, :heads], y[:, heads:-kv], y[:, -kv:], positions, slot_mapping, k_cache, v_cache,
            cos_sin,
        )[0]
    q = torch.empty(x.shape[0], heads, d, dtype=x.dtype, device=x.device)
    _C.rope_cache(q, None, None, positions, slot_mapping, k_cache, v_cache, cos_sin, y)
    return q


def rope_and_cache(q, k, v, positions, slot_mapping, k_cache, v_cache, cos_sin):
    _C.rope_cache(q, k, v, positions, slot_mapping, k_cache, v_cache, cos_sin)
    return q, k


def attention_prefill(q, k_cache, v_cache, block_table, seq_len, ctx_len, scale):
    """Single-sequence entry (tests): wrap into a one-seq batched call."""
    from ..engine.batch import FlatBatch, SeqMeta

    meta = SeqMeta(
        seq_id=0, query_len=q.shape[0], seq_len=seq_len, ctx_len=ctx_len,
        block_table=list(block_table), needs_logits=True,
    )
    dummy = torch.empty(0)
    batch = FlatBatch(
        token_ids=torch.empty(q.shape[0], device=q.device),
        positions=dummy, slot_mapping=dummy, prefills=[meta],
        num_prefill_tokens=q.shape[0], decode_seq_ids=[],
        decode_block_tables=None, decode_seq_lens=None,
        logit_rows=dummy, sample_seq_ids=[],
    )
    return attention_prefill_batch(q, k_cache, v_cache, batch, scale)


import os

_PREFILL_IMPL = os.environ.get("ACP_PREFILL_IMPL", "mfma")  # mfma | v0


def _attn_out(q):
    return torch.empty(q.shape, dtype=q.dtype, device=q.device)


def _aligned(t):
    """t, or a copy whose rows begin at multiples of 16 bytes."""
    if t.data_ptr() % 16 == 0 and t.stride(0) * t.element_size() % 16 == 0:
        return t
    return t.clone(memory_format=torch.contiguous_format)


def _attend_into(out, q, attend):
    """attend(a tensor of q's shape) into ``out``: any contiguous memory for it, or None."""
    if out is None:
        out = _attn_out(q)
    if not out.is_contiguous():
        raise RuntimeError("out must be contiguous")
    to = out if out.shape == q.shape else out.view(-1)[: q.numel()].view(q.shape)
    if to.data_ptr() % 16 == 0:
        attend(to)
    else:  # the kernels write whole units of 16 bytes
        there = _attn_out(q)
        attend(there)
        to.copy_(there)
    return out


def attention_prefill_batch(q, k_cache, v_cache, batch, scale, out=None):
    if _PREFILL_IMPL == "mfma":
        if q.shape[2] != 128:
            raise RuntimeError("prefill kernel requires head_dim 128")
        meta = batch.prefill_meta(tile_q=128)

        def attend(to):
            _C.grouped_attn(
                to, _aligned(q), k_cache, v_cache, meta.block_tables, meta.seq_lens,
                meta.ctx_lens, meta.row_starts, meta.tile_seq, meta.tile_q0, *(None,) * 6,
                scale, 0.0, _NO_WINDOW, _NO_WINDOW, 0, False, _PREFILL, 1, 1,
            )
    else:
        meta = batch.prefill_meta(tile_q=64)

        def attend(to):
            _C.prefill_attn(
                to, q, k_cache, v_cache, meta.block_tables, meta.seq_lens, meta.ctx_lens,
                meta.row_starts, meta.tile_seq, meta.tile_q0, scale,
            )
    return _attend_into(out, q, attend)


def attention_decode_batch(q, k_cache, v_cache, batch, scale, out=None):
    return _attention_decode(
        q, k_cache, v_cache, batch.decode_tables_i32(), batch.decode_lens_i32(), scale, out
    )


def attention_decode_raw(q, k_cache, v_cache, block_tables, seq_lens, scale):
    return _attention_decode(
        q, k_cache, v_cache, block_tables.int().contiguous(), seq_lens.int().contiguous(), scale
    )


def _attention_decode(q, k_cache, v_cache, tables, seq_lens, scale, out=None):
    if q.shape[2] != 128:
        raise RuntimeError("decode kernel requires head_dim 128")
    if q.shape[1] > 8 * k_cache.shape[2]:
        raise RuntimeError("GQA group must be <= 8")
    return _attend_into(out, q, lambda to: _grouped_decode(
        to, _aligned(q), k_cache, v_cache, tables, seq_lens, None, None, None, scale, 0.0,
        _NO_WINDOW, _NO_WINDOW, 0, False,
    ))


def gemm_bf16(x, w):
    out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
    _C.gemm_bf16(out, x.contiguous(), w)
    return out


def linear(x, w, bias=None, unit="plain", form=(0.0, 0.0, 0.0, 0.0), out=None, tile=-1, splits=1):
    """csrc/linear.hip; ``tile`` and ``splits`` as it chooses them unless given."""
    if out is None:
        outs = w.shape[0] // (1 if unit == "plain" else 2)
        out = torch.empty((x.shape[0], outs), dtype=x.dtype, device=x.device)
    _C.linear(out, x, w, bias, unit, *form, tile, splits)
    return out


def step_linear(x, w, bias=None, glu=False):
    out = torch.empty((x.shape[0], w.shape[0] >> glu), dtype=x.dtype, device=x.device)
    _C.step_linear(out, x, w, bias, glu)
    return out


def swiglu(gate_up):
    inter = gate_up.shape[-1] // 2
    out = torch.empty(
        (*gate_up.shape[:-1], inter), dtype=gate_up.dtype, device=gate_up.device
    )
    _C.swiglu(out, gate_up)
    return out


# ------------------------------------------------ fp32-residual norms, GLU, gates


def layernorm(x, weight, eps: float, dtype):
    out = torch.empty(x.shape, dtype=dtype, device=x.device)
    _C.residual_norm(
        x, None, None, weight, out, eps, True, 0.0, 1.0, None, None, None, 0, None, None, None,
        None, None,
    )
    return out


def residual_norm(x, y, eps: float, y_norm=None, x_norm=None, out=None, center=True,
                  offset=0.0, mult=1.0, depth=None, layer=0, x_norm2=None, out2=None,
                  experts=None, gate=None):
    states, coef, partial = depth or (None, None, None)
    rows, weights = experts or (None, None)
    _C.residual_norm(
        x, y, y_norm, x_norm, out, eps, center, offset, mult, states, coef, partial, layer,
        x_norm2, out2, rows, weights, gate,
    )


def embed_positions(token_ids, positions, table, cos_sin, x, copy=None, scale=1.0):
    _C.embed_positions(x, copy, token_ids, positions, table, cos_sin, scale)


def softcap(logits, cap):
    out = torch.empty(logits.shape, dtype=torch.float32, device=logits.device)
    _C.softcap(out, logits, cap)
    return out


def clamped_glu(gate_up, limit: float, alpha: float, offset: float, out, cubic=0.0):
    _C.clamped_glu(out, gate_up, limit, alpha, offset, cubic)


#: up to this many tokens the fused side_gate kernel beats the GEMM route
_SIDE_GATE_TOKENS = 256


def side_gate(x, y, gate, token_ids, table, offset: int):
    from . import linear

    if x.shape[0] <= _SIDE_GATE_TOKENS and x.shape[1] % 8 == 0:
        s = torch.empty(x.shape[0], gate.shape[0], dtype=gate.dtype, device=x.device)
        x_new = torch.empty_like(x)
        _C.side_gate(s, x_new, x, y, gate, token_ids, table, offset)
        return x_new, s
    xt = None if gate.dtype == torch.float32 else torch.empty_like(y)
    _C.add_to_residual(x, y, xt)
    s = linear(x if xt is None else xt, gate)
    _C.gelu_gate(s, token_ids, table, offset)
    return x, s


def side_layer_fits(x, gate, *weights) -> bool:
    """What the one launch takes, and where it is the faster: a token's workgroup reads both weights by
    itself, which is its time once they are over 256 KB each.  Us in one launch and in three, without the sum of the
    parts, of 1, 40, 128 and 512 tokens: 2048 x 64 9.8 and 10.0, 10.2 and 11.9, 10.4 and 13.9, 20.6 and 27.8.
    Twice that is faster or slower by width and tokens: 4096 x 64 15.5 and 12.9, 16.0 and 14.8, 16.5 and
    17.5, 33.9 and 43.0; 2048 x 128 14.8 and 10.1, 15.4 and 13.0, 15.9 and 16.5, 34.5 and 28.2; 8192 x 32 16.3 and
    17.3, 17.1 and 18.9, 17.9 and 20.7, 37.6 and 48.2.  4096 x 128 25.5 and 13.1, 26.2 and 16.0, 26.7 and 21.1, 58.7
    and 43.9."""
    (n, w), dim = x.shape, gate.shape[0]
    return (
        0 < n <= 512 and w % 8 == 0 and w <= 8192 and dim % 8 == 0 and dim <= 128
        and 0 < w * dim <= 1 << 17
        and all(
            t.dtype == torch.bfloat16 and t.is_contiguous() and t.data_ptr() % 16 == 0
            for t in (gate, *weights)
        )
    )


def side_layer(x, y, gate, token_ids, table, offset: int, proj, eps: float, y_norm, x_norm, out):
    _C.side_layer(x, y, gate, token_ids, table, offset, proj, eps, y_norm, x_norm, out)


# ------------------------------------------------------------ latent attention

_NO_WINDOW = 1 << 30
_MAX_SPLIT = 32


def latent_inputs(kv, norm_w, eps: float, kv_rank: int, rot_dim: int, rank: int,
                  positions, slot_mapping, cos_sin, cache, q=None, q_norm=None, q_rank=0, glu=None):
    cq = None if q is None else torch.empty(q.shape, dtype=q.dtype, device=q.device)
    _C.latent_inputs(
        cache, kv, norm_w, positions, slot_mapping, cos_sin, eps, kv_rank, rot_dim, rank,
        cq, q, q_norm, q_rank, *(glu or (None, None, 0.0, 0.0, 0.0)),
    )
    return cq


def head_linear(x, w, out, gate=None):
    _C.head_linear(out, x, w, gate)
    return out


def _latent_attn(out, q, q_rot, cos_sin, rot_dim, cache, tables, seq_lens, prefill, tiles,
                 mg, max_keys, scale, window, mfma, sink, merge=True):
    """One launch over prefill tiles (prefill = their metadata) or decode
    rows.  Few tiles split their keys over several workgroups; without ``merge`` their parts stay so and are
    returned, with their sums, the most that a row can have and the number that most have."""
    n_split = 1
    if mfma:
        keys = min(max_keys, window)
        most = min(_MAX_SPLIT, -(-keys // 128))
        # workgroups that fill the chip: the tiles of a wide latent take a CU's LDS
        wide = q.shape[2] >= 256
        n_split = max(1, min(most, (256 if wide else 512) // tiles))
        # Or half of it for up to 16 rows, by smaller tiles, which pays for parts of 320 keys, or 768
        # undivided, from 16 sequences on.  16 heads of rank 512, us by up to 256 workgroups and 512: 12 x
        # 7500 31.1 and 32.8, 16 x 8000 38.8 and 35.5, 32 x 2000 of 250 keys a part 26.1 and 28.7, 40 x
        # 2000 of 333 35.5 and 34.0, 64 x 4200 71 and 65; undivided 190 x 500 32.5 and 36.0, x 1000 56.4 and
        # 53.4, 129 x 2000 98 and 64.  More workgroups than 512 gain nothing: 40 x 200 to 6000, a step's 20
        # layers, 2400 by 512 and 2455 by 1024
        if wide and mg == 1 and 16 <= tiles <= 256 and keys >= (320 * n_split if n_split > 1 else 768):
            n_split = max(1, min(most, 512 // tiles))
    part = ml = None
    cap = n_split
    if n_split > 1:
        # Decode rows' parts by length, a long row's up to three times as many: us of 16 heads of rank 512 with
        # the product behind, by as many parts a row, and so: 40 x 200 to 6000 51.0 and 44.0, 8000 beside 39 x
        # 500 53.6 and 30.8, 100 x 500 to 3000 60.4 and 52.4, 4000 beside 249 x 800 131 and 68; alike 40 x 2000
        # 35.9 and 34.3, 250 x 1000 66.6 and 66.9, 130 x 1000 46.6 and 48.4, as every workgroup reads all lengths.
        # Not where a window makes most of them alike, 24 x 300 to 1500 by 1024 21.3 and 23.1
        if prefill is None and tables.shape[0] <= 256 and window >= max_keys:
            cap = max(n_split, min(most, 3 * n_split))
        rows = q.shape[0] * q.shape[1]
        part = torch.empty(cap * rows * q.shape[2], dtype=torch.float32, device=q.device)
        # rows no tile covers (skipped chunks) must merge to nothing
        new = torch.empty if prefill is None else torch.zeros
        ml = new(2 * cap * rows, dtype=torch.float32, device=q.device)
    # The product takes so many parts of a narrow latent one after another, longer than a launch: one sequence
    # in 32 of them, us merged by itself and in the product: 8 heads of rank 64 12.8 and 13.3, 32 of 128 16.7
    # and 17.6, 16 of 256 16.2 and 16.3, but of 512 22.6 and 21.3; four in 16: 11.3 and 10.7, 15.0 and 14.6
    merge = merge or n_split > 16 and q.shape[2] <= 256
    m = prefill
    _C.latent_attn(
        out, q, q_rot, cos_sin, rot_dim, cache, tables, seq_lens,
        *((m.ctx_lens, m.row_starts, m.tile_seq, m.tile_q0) if m else (None,) * 4),
        part, ml, sink, scale, window, mg, n_split, cap, mfma, merge,
    )
    return None if merge or n_split == 1 else (part, ml, cap, n_split)


def latent_attention(q, q_rot, cos_sin, rot_dim: int, cache, batch, scale: float, window,
                     row0: int = 0, skip=(), sink=None):
    return _latent_rows(
        q, q_rot, cos_sin, rot_dim, cache, batch, scale, window, row0, skip, sink, True
    )[0]


def latent_values(q, q_rot, cos_sin, rot_dim: int, cache, batch, scale: float, window,
                  row0: int, skip, sink, w, out, gate):
    latent, parts = _latent_rows(
        q, q_rot, cos_sin, rot_dim, cache, batch, scale, window, row0, skip, sink, False
    )
    if parts is None:
        return head_linear(latent, w, out, gate)
    P = q.shape[0] - batch.num_decode
    if P:
        head_linear(latent[:P], w, out[:P], None if gate is None else gate[:P])
    _C.merge_head_linear(out[P:], *parts, w, None if gate is None else gate[P:])
    return out


def _latent_rows(q, q_rot, cos_sin, rot_dim, cache, batch, scale, window, row0, skip, sink, merge):
    """latent_attention(), and the decode rows' parts if these are not merged."""
    from . import LATENT_RANKS

    parts = None
    N, H, rank = q.shape
    out = torch.empty(N, H, rank, dtype=q.dtype, device=q.device)
    window = window or _NO_WINDOW
    mfma = q.dtype == torch.bfloat16 and rank in LATENT_RANKS and q_rot.shape[2] == 64
    most = 4 if rank <= 256 else 2
    P = batch.num_prefill_tokens - row0
    common = (cos_sin, rot_dim, cache)
    chunks = tuple(i for i in range(len(batch.prefills)) if i not in skip)
    if chunks:
        meta = batch.prefill_meta(
            16 * most if mfma else 1, rows_per_token=H, only=chunks, row_base=row0
        )
        _latent_attn(
            out[:P], q[:P], q_rot[:P], *common, meta.block_tables, meta.seq_lens, meta,
            meta.tile_seq.numel(), most, max(batch.prefills[i].seq_len for i in chunks),
            scale, window, mfma, sink,
        )
    if batch.num_decode:
        mg = 1 if H <= 16 else 2 if H <= 32 else most
        tables = batch.decode_tables_i32()
        parts = _latent_attn(
            out[P:], q[P:], q_rot[P:], *common, tables, batch.decode_lens_i32(), None,
            batch.num_decode * -(-H // (16 * mg)), mg,
            tables.shape[1] * cache.shape[1], scale, window, mfma, sink, merge,
        )
    return out, parts


#: expanded keys and values built at a time
_EXPAND_BYTES = 2 << 30


def can_expand(dtype, d: int, v: int, rot: int) -> bool:
    from . import LATENT_HEADS

    return dtype == torch.bfloat16 and rot == 64 and d in LATENT_HEADS and v in LATENT_HEADS


def _expansion_groups(batch, chunks, window: int, bytes_per_key: int):
    groups, at = [], 0
    for i in chunks:
        m = batch.prefills[i]
        keys = (m.seq_len - max(0, m.ctx_len - window + 1)) * bytes_per_key
        if not groups or at + keys > _EXPAND_BYTES:
            groups.append([])
            at = 0
        groups[-1].append(i)
        at += keys
    return [tuple(g) for g in groups]


def latent_expanded_prefill(q, w_ukv, gate, cos_sin, rot_dim: int, cache, batch, chunks,
                            rank: int, scale: float, window, out, sink=None):
    from . import linear

    window = window or _NO_WINDOW
    row = cache.shape[2]
    groups = batch.memo(
        ("expansion_groups", chunks, window, w_ukv.shape[0]),
        lambda: _expansion_groups(batch, chunks, window, 2 * w_ukv.shape[0]),
    )
    for group in groups:
        meta = batch.prefill_meta(128, only=group, window=window)
        rows = torch.empty(meta.num_keys, row, dtype=q.dtype, device=q.device)
        _C.latent_gather(
            rows, cache, meta.block_tables, meta.seq_lens, meta.key_first, meta.key_starts,
            meta.max_keys,
        )
        _C.latent_prefill(
            out, q, linear(rows[:, :rank], w_ukv), rows[:, rank:], gate, cos_sin, rot_dim,
            meta.seq_lens, meta.ctx_lens, meta.row_starts, meta.tile_seq, meta.tile_q0,
            meta.key_first, meta.key_starts, sink, scale, window,
        )


# ---------------------------------------- grouped attention: caps, windows, sinks

_PLAIN, _DECODE, _PREFILL, _TALK_DECODE, _TALK_PREFILL = range(5)


def cache_keys_values(k, v, slot_mapping, k_cache, v_cache):
    _C.cache_keys_values(k_cache, v_cache, k, v, slot_mapping)


def _conv_rows(batch):
    """Per row of a step: rows of its sequence right before it, and its state slot.
    None, slots: every row is alone in its sequence's step."""
    if not batch.prefills:
        return None, batch.decode_state_slots
    P, meta = batch.num_prefill_tokens, batch.prefill_meta(16)
    ctx, slots = torch.stack([meta.ctx_lens, meta.state_slots]).repeat_interleave(
        meta.seq_lens - meta.ctx_lens, 1, output_size=P
    )
    back = batch.positions[:P].int() - ctx
    if batch.num_decode:
        back = torch.cat([back, back.new_zeros(batch.num_decode)])
        slots = torch.cat([slots, batch.decode_state_slots])
    return back, slots.contiguous()


def _ring_rows(batch, taps: int):
    """The last rows of every portion, as many as a ring holds."""
    rows, at = [], 0
    for m in batch.prefills:
        at += m.query_len
        rows.extend(range(at - min(m.query_len, taps), at))
    rows.extend(range(at, at + batch.num_decode))
    if batch._stager is not None:
        return batch._stager.tensor(f"ring_rows{taps}", rows, "int32")
    return torch.tensor(rows, dtype=torch.int32, device=batch.positions.device)


def attention_inputs(proj, heads, dim, vdim, k_cache, v_cache, batch, eps, conv, ring, q_norm,
                     k_norm, v_norm, cos_sin, head_mult, q_temp):
    q = torch.empty(proj.shape[0], heads, k_cache.shape[3], dtype=proj.dtype, device=proj.device)
    back = states = ring_rows = None
    if conv is not None:
        back, states = batch.memo("conv_rows", lambda: _conv_rows(batch))
        if batch.prefills:
            taps = conv.shape[0]
            ring_rows = batch.memo(("ring_rows", taps), lambda: _ring_rows(batch, taps))
    coef, every = q_temp or (0.0, 0.0)
    _C.attention_inputs(
        q, k_cache, v_cache, proj, batch.positions, batch.slot_mapping, dim, vdim, eps, conv,
        ring, back, states, ring_rows, ring_rows is None, q_norm, k_norm, v_norm, cos_sin,
        head_mult, coef, every,
    )
    return q


def _grouped_decode(out, q, k_cache, v_cache, tables, seq_lens, sink, bias, gate, scale, cap,
                    window, chunk, keep_first, sigmoid):
    """One token per sequence, head sizes of the matrix-core kernels.  Grid and workspace
    depend on sizes alone, not on the lengths, so that a step can be captured."""
    (B, H, d), v, G = q.shape, out.shape[2], k_cache.shape[2]
    gm = next((n for n in (1, 2, 4) if n >= H // G), 8)  # query heads a workgroup holds
    # workgroups that fill the chip at once
    keys = min(tables.shape[1] * k_cache.shape[1], window + keep_first, chunk)
    groups = G * -(-(H // G) // gm)
    pieces, part, ml = 0, None, None
    if B * groups < _WHOLE_GROUPS and keys > 128:
        pieces = max(1, _DECODE_GROUPS // groups)
        part = torch.empty(2 * (2 * pieces + B) * H * v, dtype=torch.float32, device=q.device)
        ml = torch.empty(4 * (2 * pieces + B) * H, dtype=torch.float32, device=q.device)
    _C.grouped_attn(
        out, q, k_cache, v_cache, tables, seq_lens, None, None, None, None, sink, bias, gate,
        None, part, ml, scale, cap, window, chunk, keep_first, sigmoid, _DECODE, gm, pieces,
    )


#: workgroups that share a decode step's keys: the 2 a CU that fit
_DECODE_GROUPS = 512
#: from so many sequences and key heads on a sequence is one workgroup's (of 8 heads 190 x 700 to 1300 keys: 141
#: us, in even shares 144 with the merge; 256 x 1024 174 and 194; 230 x 500 to 3500 331 and 326).  The host
#: does not see the lengths: where one sequence is by far the longest that is the slower choice (129 x 300
#: keys and one of 8000: 155 and 58 us)
_WHOLE_GROUPS = 1024


def grouped_attention(q, k_cache, v_cache, batch, scale: float, cap, window, keep_first: int,
                      sink, out, bias=None, sigmoid=False, gate=None, chunk=None, talk=None):
    from . import LATENT_HEADS

    H, d, v, G = q.shape[1], q.shape[2], out.shape[2], k_cache.shape[2]
    rest = (scale, cap or 0.0, window or _NO_WINDOW, chunk or _NO_WINDOW, keep_first, sigmoid)
    bf16 = q.dtype == torch.bfloat16
    if talk is None:
        tiled = bf16 and d in LATENT_HEADS and v in LATENT_HEADS and not (sigmoid and cap)
        kinds, tile = ((_DECODE, _PREFILL) if tiled else (_PLAIN, _PLAIN)), 128
    else:
        tiled = bf16 and not (sigmoid or cap or keep_first) and all(
            t is None for t in (sink, bias, gate))
        tile = _C.talk_prefill_tokens(H, G, d, v, k_cache.shape[1]) if tiled else 0
        tiled = tiled and _C.talk_decode_fits(H, G, d, v)
        kinds = (_TALK_DECODE if tiled else _PLAIN, _TALK_PREFILL if tile else _PLAIN)
    P = batch.num_prefill_tokens

    def gates(r):
        return None if gate is None else gate[r]

    if batch.prefills:
        if kinds[1] == _TALK_PREFILL:
            meta = batch.prefill_meta(tile, chunk=chunk or _NO_WINDOW)
        else:
            meta = batch.prefill_meta(1 if kinds[1] == _PLAIN else tile)
        _C.grouped_attn(
            out[:P], q[:P], k_cache, v_cache, meta.block_tables, meta.seq_lens, meta.ctx_lens,
            meta.row_starts, meta.tile_seq, meta.tile_q0, sink, bias, gates(slice(0, P)), talk,
            None, None, *rest, kinds[1], 1, 1,
        )
    if not batch.num_decode:
        return
    tables, rows = batch.decode_tables_i32(), batch.num_decode * H
    if kinds[0] == _DECODE:
        _grouped_decode(
            out[P:], q[P:], k_cache, v_cache, tables, batch.decode_lens_i32(), sink, bias,
            gates(slice(P, None)), *rest,
        )
        return
    n_split, part, ml = 1, None, None
    if kinds[0] == _TALK_DECODE:  # a workgroup has all heads, and 4 waves with 32 keys each
        keys = min(tables.shape[1] * k_cache.shape[1], rest[2], rest[3])  # a row may see
        n_split = max(1, min(_MAX_SPLIT, 1024 // batch.num_decode, -(-keys // 128)))
    if n_split > 1:
        part = torch.empty(n_split * rows * v, dtype=torch.float32, device=q.device)
        ml = torch.empty(2 * n_split * rows, dtype=torch.float32, device=q.device)
    _C.grouped_attn(
        out[P:], q[P:], k_cache, v_cache, tables, batch.decode_lens_i32(), None, None, None,
        None, sink, bias, gates(slice(P, None)), talk, part, ml, *rest,
        kinds[0], 1, n_split,
    )


# -------------------------------------------------------------------- experts


def moe_route(h, router, bias, top: int, sigmoid=False, scale=1.0):
    ids = torch.empty(h.shape[0], top, dtype=torch.int32, device=h.device)
    weights = torch.empty(h.shape[0], top, dtype=torch.float32, device=h.device)
    _C.moe_route(ids, weights, h, router, bias, sigmoid, scale)
    return ids, weights


#: average rows per expert from which the tiled product is faster (its weights are read
#: once, however many rows there are)
_TILED_ROWS = 12


def moe_experts(h, gate_up, down, ids, glu):
    (N, k), E, inner = ids.shape, gate_up.shape[0], down.shape[2]
    if N * h.stride(0) >= 1 << 30 and N > 1:  # the tiled product's offsets have 32 bits
        halves = [slice(0, N // 2), slice(N // 2, N)]
        return torch.cat([moe_experts(h[r], gate_up, down, ids[r], glu) for r in halves])
    n, device = N * k, h.device
    act = torch.empty(n, inner, dtype=h.dtype, device=device)
    rows = torch.empty(N, k, down.shape[1], dtype=h.dtype, device=device)
    form = (glu.limit, glu.alpha, glu.offset, glu.cubic)
    perm = offsets = tile_expert = tile_row = None
    kind, tt = 0, 1
    if h.dtype == torch.bfloat16:
        tiled = (
            n >= _TILED_ROWS * E and gate_up.shape[2] % 128 == 0 and inner % 128 == 0
            and max(gate_up[0].numel(), down[0].numel()) < 1 << 30
        )
        kind, tt = (2, 1) if tiled else (1, 1 if n <= 8 * E else 2)
        perm = torch.empty(n, dtype=torch.int32, device=device)
        offsets = torch.empty(E + 2, dtype=torch.int32, device=device)
        if tiled:
            tiles = torch.empty(2, n // _C.EXPERT_TILE + E, dtype=torch.int32, device=device)
            tile_expert, tile_row = tiles
        _C.moe_group(perm, offsets, tile_expert, tile_row, ids, E)
    grouped = (ids, perm, offsets, tile_expert, tile_row)
    _C.experts_linear(act, h, gate_up, *grouped, True, *form, kind, tt)
    _C.experts_linear(rows.view(n, -1), act, down, *grouped, False, *form, kind, tt)
    return rows


# ----------------------------------------------------------------- delta rule


def _step_threads(D: int, V: int, workgroups: int) -> int:
    """Threads of a decode workgroup: at most 16 rows of the state per thread, fewer
    while the workgroups do not fill the chip."""
    columns = V // 4 if V % 4 == 0 else V
    rows = 16 if workgroups >= 512 else 4
    for n in (256, 512):
        if n >= columns and n // columns * rows >= D:
            return n
    return 1024


def _scan_columns(prefills, columns: int) -> int:
    """Columns of the state a lane works on.  Two take less work a token, one is the shorter
    chain: with two once there is work beside the longest sequence's chain.  2048 columns, one
    and two, us: 6 x 1000 tokens 381, 418; 7 x 1000 481, 430; 8 of 300 to 2600 725, 808; 11 of
    them 953, 859; 3000 and 32 x 300 810, 959."""
    lens = [m.query_len for m in prefills]
    return 2 if sum(lens) * columns > 3 * 4096 * max(lens) else 1


def _scan_in_chunks(prefills, H: int, D: int, V: int, dtype) -> int:
    """16s of columns a workgroup of the recurrence by chunks of 16 tokens, 0: token by token.  By
    chunks, heads of 128 key channels: a launch more, a shorter chain, but whole chunks of work for tokens past
    the end of a portion.  So from 49 tokens on, and where all portions' chunks are at most a third more
    work than their tokens or that is little beside the longest one's chain; and portions have 16 tokens on
    average, which bounds the workspace.  All launches of a layer with 16 heads of 128 x 128, us, token by
    token and by chunks: 17 tokens 28, 32; 33 31, 33; 64 36, 34; 12 x 64 69, 62; 20 x 49 84, 80; 24 x 300 387, 311;
    8000 1444, 631; a portion of 49 beside 8 of 17 47, 48, beside 40 of 17 91, 99, beside 40 of 1 74, 78; 600 beside
    200 x 20 354, 372; 300 beside 40 x 17 127, 113; 1000 beside 100 x 17 240, 197.  Of 320 steps of 1 to 260
    portions and 8 to 32 heads 4 take more than 2% longer than token by token, at most 3 us; where the longest portion
    alone decided 25 did, up to 42%.  In fp32 token by token: results of keys that are alike are further from 64 bits
    by chunks.
    16 columns a workgroup are the shorter chain, 32 less work beside the longest sequence's, of which a short
    portion has more than its tokens: 760 to 2140 330, 380 (3.2 times the longest one's chunks); 4 x 400 103,
    99; 8 x 1000 419, 340; 1000 beside 100 x 17 231, 197; with 32 heads 3 x 600 184, 180; 8000 795, 948."""
    lens = [m.query_len for m in prefills]
    tokens, longest = sum(lens), max(lens)
    if dtype != torch.bfloat16 or D != 128 or V % 16 or longest <= 48 or 16 * len(lens) > tokens:
        return 0
    chunks = sum(-(-n // 16) for n in lens)
    if 48 * chunks > 4 * tokens + 3 * longest:
        return 0
    beside = (chunks + len(lens)) * H * V > 4 * 2048 * (-(-longest // 16) + 1)
    return 2 if V % 32 == 0 and beside else 1


def gated_delta_bytes(tokens: int, H: int, D: int, V: int, dtype) -> int:
    """The most that the chunks of a step of so many prompt tokens take: _scan_in_chunks() lets through no more
    portions than 16s of tokens."""
    if dtype != torch.bfloat16 or D != 128 or V % 16:
        return 0
    return 4 * 2 * (tokens // 16) * H * _C.DELTA_CHUNK_FLOATS


def gated_delta(qkv, conv, b, z, A_log, dt_bias, gate, norm, eps, unit_eps, kv_heads,
                state, conv_state, batch, gate_silu=False):
    H, D, V = state.shape[1:]
    out = torch.empty(gate.shape, dtype=qkv.dtype, device=qkv.device)
    P = batch.num_prefill_tokens

    def rows(r):
        return (out[r], qkv[r], conv, b[r], z[r], A_log, dt_bias, gate[r], norm, state,
                conv_state)

    if batch.prefills:
        meta = batch.prefill_meta(16)

        def space(n, dtype=torch.float32):
            return torch.empty(P * n, dtype=dtype, device=qkv.device)

        chunks = None
        cpl = batch.memo(
            ("scan_chunks", H, D, V, qkv.dtype),
            lambda: _scan_in_chunks(batch.prefills, H, D, V, qkv.dtype),
        )
        if cpl:
            n = (P // 16 + len(batch.prefills)) * H * _C.DELTA_CHUNK_FLOATS
            chunks = torch.empty(n, device=qkv.device)
        else:
            cpl = batch.memo(("scan_columns", H * V), lambda: _scan_columns(batch.prefills, H * V))
        _C.delta_prompts(
            *rows(slice(0, P)), meta.seq_lens, meta.state_slots, kv_heads, eps, unit_eps,
            gate_silu, meta.ctx_lens, meta.row_starts, meta.tile_seq, meta.tile_q0,
            space(qkv.shape[1], qkv.dtype), space(3 * kv_heads),
            None if z.shape[1] == H else space(H * D), space(H * V), cpl, chunks,
        )
    if batch.num_decode:
        _C.delta_step(
            *rows(slice(P, None)), batch.decode_lens_i32(), batch.decode_state_slots, kv_heads,
            eps, unit_eps, gate_silu, _step_threads(D, V, batch.num_decode * H),
        )
    return out


def softmax_sample(logits, temperatures, top_ks, top_ps, gen, mask=None,
                   uniforms=None, mask_map=None):
    B, V = logits.shape
    out = torch.empty(B, dtype=torch.long, device=logits.device)
    if uniforms is None:
        uniforms = torch.rand(B, device=logits.device, generator=gen)
    if V > 512:
        # BPE-scale vocab: LDS radix-select kernel, bf16 logits unconverted
        # (csrc/sampling_fullvocab.hip); masks are compact [M, V] rows with
        # mask_map [B] indirection (-1 = unconstrained row)
        if logits.dtype not in (torch.bfloat16, torch.float32):
            logits = logits.float()
        if mask is not None and mask_map is None:
            mask_map = torch.arange(B, dtype=torch.int32, device=logits.device)
        _C.sample_fullvocab(
            out, logits.contiguous(), temperatures.float().contiguous(),
            top_ks.long().contiguous(), top_ps.float().contiguous(),
            uniforms.contiguous(),
            mask.contiguous() if mask is not None else None,
            mask_map.contiguous() if mask is not None else None,
        )
        return out
    _C.sample(
        out, logits.float().contiguous(), temperatures.float().contiguous(),
        top_ks.long().contiguous(), top_ps.float().contiguous(),
        uniforms.contiguous(), mask.contiguous() if mask is not None else None,
    )
    return out
