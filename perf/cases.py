"""The work that users of the framework have it do, as cases that can be timed and checked.

Most cases are steps of the serving engine on whole models with random weights: the
scheduler lays sequences out in pages, and a pass is ``InferenceEngine.forward_batch`` on
their batch, from token ids to logits.  Sequences have ragged, mostly odd lengths, and pages
of sequences that grew side by side alternate in the pool, as they do in service.  The batch
keeps what the scheduler uploads for a step; what the kernels derive from it is made in every
pass, as in service, where every step's batch is new.

The other cases are the two parts of a step that cannot be compared through a whole model:
the mixture of experts, because a rounding that moves a token to another expert changes all
that follows, and the sampler, whose tokens are whole numbers.

A case is plain values, all sizes follow from them (not from the seed), and
everything random follows from the seed.
"""
import dataclasses
import gc
import math

import torch

from agentcontrolplane_amd import ops
from agentcontrolplane_amd.engine.config import PRESETS, EngineConfig
from agentcontrolplane_amd.engine.engine import InferenceEngine
from agentcontrolplane_amd.engine.request import InferenceRequest, SamplingParams
from agentcontrolplane_amd.models.experts import Experts

DEVICE = "cuda"
BLOCK = EngineConfig.kv_block_size

#: per model: tokens of the page pool, which holds three states and what replaces one of
#: them, and sequences at a time
POOLS = {
    "llama3-8b": (800_000, 1024),
    "llama2-7b": (120_000, 256),
    "fetolix-2b": (600_000, 512),
    "tezinex-2b": (60_000, 64),
}
#: the most tokens that a state of these models caches
MOST_TOKENS = {name: tokens // 4 for name, (tokens, _) in POOLS.items()}


def _step(name, model, *, chunks=(0, 0, 0), cached=(0, 0), rows=(0, 0, 0), then_decode=False):
    """An engine step: ``chunks`` (count, shortest, longest) prompt chunks behind ``cached``
    (least, most) tokens, and ``rows`` (count, least, most cached tokens) of one token each.
    ``then_decode``: the chunks' sequences take one token each in a second step."""
    return {
        "name": name, "kind": "step", "model": model,
        "chunks": chunks[0], "chunk_lo": chunks[1], "chunk_hi": chunks[2],
        "cached_lo": cached[0], "cached_hi": cached[1],
        "rows": rows[0], "row_lo": rows[1], "row_hi": rows[2], "then_decode": then_decode,
    }


def listed():
    return [
        # one user's answer being written, late in a long conversation: latency
        _step("llama_decode_one", "llama3-8b", rows=(1, 4001, 4001)),
        # a few dozen conversations of all lengths
        _step("llama_decode_ragged", "llama3-8b", rows=(61, 310, 4000)),
        # the agent loop's decode steps: many tasks, each about a system prompt and a turn long
        _step("llama_decode_wave", "llama3-8b", rows=(190, 700, 1300)),
        # a model whose heads all have keys of their own
        _step("mha_decode", "llama2-7b", rows=(13, 300, 3900)),
        # tool results come back as short chunks on cached prefixes while other tasks decode
        _step("llama_tool_turns", "llama3-8b", chunks=(9, 35, 310), cached=(790, 1500),
              rows=(120, 700, 1400)),
        # the agent loop's prompts: one step of the default token budget
        _step("llama_prompt_wave", "llama3-8b", chunks=(15, 700, 1400)),
        # one long document
        _step("llama_prompt_long", "llama3-8b", chunks=(1, 8131, 8131)),
        # cached latents instead of keys and values
        _step("latent_decode", "fetolix-2b", rows=(40, 200, 6000)),
        # recurrent layers: prompts, then the first token of each answer from the kept states
        _step("delta_prompts", "tezinex-2b", chunks=(5, 300, 2600), then_decode=True),
        # the experts of a decode step, and of a step of prompts
        {"name": "experts_decode", "kind": "experts", "model": "lobuvik-8b", "tokens": 48},
        {"name": "experts_prompt", "kind": "experts", "model": "lobuvik-8b", "tokens": 4093},
        # a step's tokens from the whole vocabulary of a tokenizer
        {"name": "sample", "kind": "sample", "vocab": 128256, "tokens": 190},
    ]


def _log_int(rng, lo, hi):
    """Even over the logarithm, odd as often as even."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _sorted_pair(rng, lo, hi):
    return sorted((_log_int(rng, lo, hi), _log_int(rng, lo, hi)))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "chunks", "prompts", "prompts", "latent",
                       "delta", "experts", "sample"])
    if kind == "decode":
        model = rng.choice(["llama3-8b", "llama3-8b", "llama2-7b"])
        most = min(8000, PRESETS[model].max_position - 96)
        lo, hi = _sorted_pair(rng, 100, most)
        n = _log_int(rng, 1, max(1, min(230, MOST_TOKENS[model] // (hi + BLOCK))))
        case = _step("", model, rows=(n, lo, hi))
    elif kind == "chunks":
        new, old = _sorted_pair(rng, 17, 700), _sorted_pair(rng, 60, 3000)
        rows = (_log_int(rng, 1, 150), *_sorted_pair(rng, 100, 1300))
        case = _step("", "llama3-8b", chunks=(_log_int(rng, 1, 12), *new), cached=old, rows=rows)
    elif kind == "prompts":
        model = rng.choice(["llama3-8b", "llama3-8b", "llama2-7b"])
        lo, hi = _sorted_pair(rng, 33, 3900 if model == "llama2-7b" else 8000)
        n = _log_int(rng, 1, max(1, min(64, 10000 // hi)))
        case = _step("", model, chunks=(n, lo, hi))
    elif kind == "latent":
        lo, hi = _sorted_pair(rng, 100, 7000)
        case = _step("", "fetolix-2b", rows=(
            _log_int(rng, 1, min(64, MOST_TOKENS["fetolix-2b"] // (hi + BLOCK))), lo, hi))
    elif kind == "delta":
        lo, hi = _sorted_pair(rng, 50, 3000)
        n = _log_int(rng, 1, max(1, min(12, 8000 // hi)))
        case = _step("", "tezinex-2b", chunks=(n, lo, hi), then_decode=True)
    elif kind == "experts":
        case = {"kind": "experts", "model": rng.choice(["lobuvik-8b", "lobuvik-2b"]),
                "tokens": _log_int(rng, 1, 4093)}
    else:
        case = {"kind": "sample", "vocab": rng.choice([32000, 128256, 152064]),
                "tokens": _log_int(rng, 1, 512)}
    case.pop("name", None)
    return case


def _spread(n, lo, hi):
    """n whole numbers over [lo, hi], in no order."""
    return [lo + round((hi - lo) * ((0.5 + i * 0.6180339887) % 1)) for i in range(n)]


def _lengths(case):
    """[(cached tokens, new tokens)]: the chunks, then the rows."""
    new = _spread(case["chunks"], case["chunk_lo"], case["chunk_hi"])
    old = _spread(case["chunks"], case["cached_lo"], case["cached_hi"])
    rows = _spread(case["rows"], case["row_lo"], case["row_hi"])
    return list(zip(old, new)) + [(c, 1) for c in rows]


# ------------------------------------------------------------------- preparation

_engine = None  # the last one asked for: a program keeps its weights and page pool


def _engine_of(model):
    global _engine
    if _engine is None or _engine.cfg.model != model:
        _engine = None
        gc.collect()
        torch.cuda.empty_cache()
        tokens, sequences = POOLS[model]
        _engine = InferenceEngine(
            EngineConfig(
                model=model, device=DEVICE, num_kv_blocks=tokens // BLOCK,
                max_batch_size=sequences, num_state_slots=sequences,
            ),
            start=False,
        )
        # an ended sequence's pages are given back
        _engine.scheduler.continuation_cache = False
        m = _engine.model
        if not _engine.mcfg.layers:
            # a plain random start multiplies every rounding by its depth; with an embedding
            # of unit size and smaller results, layers add to the residual about as a
            # trained model's do
            m.embed.mul_(50.0)
            for layer in m.layers:
                layer.o.mul_(1 / 16)
                layer.down.mul_(1 / 16)
    return _engine


class Steps:
    """Sequences in an engine's pages, and the batches of one or two steps on them."""

    def __init__(self, case, seed):
        self.engine = engine = _engine_of(case["model"])
        sched, g = engine.scheduler, torch.Generator(DEVICE).manual_seed(seed)
        lengths = _lengths(case)
        extra = 1 if case["then_decode"] else 0
        ids = torch.randint(
            0, engine.mcfg.vocab_size, (sum(c + n + extra for c, n in lengths),), generator=g,
            device=DEVICE,
        ).tolist()
        self.seqs, self.ids, at = [], [], 0
        for cached, new in lengths:
            self.ids.append(ids[at : at + cached + new + extra])
            at += cached + new + extra
            self.seqs.append(sched.add_request(
                InferenceRequest(self.ids[-1][: cached + new], SamplingParams(max_tokens=1))
            ))
        for s in self.seqs:
            sched.waiting.remove(s)
            sched.running.append(s)
            sched.reserve(s)
        grown = 0
        while any(grown < cached for cached, _ in lengths):
            for s, (cached, _) in zip(self.seqs, lengths):
                if grown < cached:
                    engine.bm.append_tokens(s.seq_id, min(4 * BLOCK, cached - grown))
            grown += 4 * BLOCK
        for s, (cached, _) in zip(self.seqs, lengths):
            s.num_processed = cached
        self.lengths, self.batches = lengths, []
        self._plan([(s, new, [new - 1]) for s, (_, new) in zip(self.seqs, lengths)])
        if extra:
            for s, mine in zip(self.seqs, self.ids):
                s.prompt_ids.append(mine[-1])
            self._plan([(s, 1, [0]) for s in self.seqs])
        self.tables = [list(engine.bm.block_table(s.seq_id)) for s in self.seqs]
        pages = torch.tensor(sum(self.tables, []), device=DEVICE)
        for cache in self.caches():
            # as the models' own rows: a projection of a normed row by weights of 0.02
            std = 0.02 * engine.mcfg.hidden_size ** 0.5
            rows = torch.randn(
                len(pages), *cache.shape[1:], generator=g, device=DEVICE, dtype=cache.dtype
            )
            cache[pages] = rows.mul_(std)

    def caches(self):
        m = self.engine.model
        return getattr(m, "caches", None) or m.k_caches + m.v_caches

    def _plan(self, portions):
        self.batches.append(self.engine.scheduler.schedule_portions(portions)[0])

    def cached(self, cache, n):
        """Sequence n's rows of a cache ahead of the step, in 64 bits."""
        rows = cache[torch.tensor(self.tables[n], device=DEVICE)].flatten(0, 1)
        return rows[: self.lengths[n][0]].double()

    def run(self):
        out = []
        for batch in self.batches:
            logits = self.engine.forward_batch(dataclasses.replace(batch, _memo=None))
            out.append(logits)
        return out

    def __del__(self):
        for s in getattr(self, "seqs", ()):
            self.engine.scheduler.finish_seq(s, "stop")


class ExpertLayer:
    """One layer's experts and the normed rows that reach them."""

    def __init__(self, case, seed):
        cfg = PRESETS[case["model"]]
        self.spec = next(x.mlp for x in cfg.layers if hasattr(x.mlp, "experts"))
        self.width = cfg.hidden_size
        g = torch.Generator(DEVICE).manual_seed(seed)
        self.layer = Experts(self.spec, self.width, 0, 1)
        shapes = dict(self.layer.shapes())

        def get(name):
            t = torch.empty(shapes[name], dtype=torch.bfloat16, device=DEVICE)
            return t.normal_(0.0, 0.02, generator=g)

        self.layer.load(get, "")
        self.h = torch.randn(
            case["tokens"], self.width, generator=g, device=DEVICE, dtype=torch.bfloat16
        )

    def run(self):
        return self.layer.forward(self.h)


class Sampler:
    """A step's logits and its requests' sampling parameters: plain draws, top-k,
    nuclei and a few greedy ones, each with a random number of its own."""

    def __init__(self, case, seed):
        n, g = case["tokens"], torch.Generator(DEVICE).manual_seed(seed)
        self.logits = torch.randn(n, case["vocab"], generator=g, device=DEVICE) * 2.5
        i = torch.arange(n, device=DEVICE)
        self.temperatures = torch.where(i % 8 == 7, 0.0, 0.8)
        self.top_ks = torch.where(i % 4 == 1, 50, 0)
        self.top_ps = torch.where(i % 4 == 2, 0.95, 1.0)
        self.uniforms = torch.rand(n, generator=g, device=DEVICE)

    def run(self):
        return ops.softmax_sample(
            self.logits, self.temperatures, self.top_ks, self.top_ps, None,
            uniforms=self.uniforms,
        )


KINDS = {"step": Steps, "experts": ExpertLayer, "sample": Sampler}


def prepare(case, seed):
    return KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# -------------------------------------------------------------------------- work


def _work_step(case):
    cfg = PRESETS[case["model"]]
    lengths, vocab, width = _lengths(case), cfg.vocab_size, cfg.hidden_size
    tokens, logits = sum(n for _, n in lengths), len(lengths)
    runs = [cfg.layers[i] for i, _ in cfg.layer_runs] if cfg.layers else []
    head = vocab * width
    # weights every token passes: each read once
    weights = cfg.params_bytes(1) - head * (1 if cfg.tie_embeddings else 2)
    if cfg.token_side_dim:
        weights -= vocab * cfg.token_side_dim * len(cfg.layers)
    passed = weights  # a looped layer's count in every pass
    if cfg.loop:
        again = sum(
            x.mixer.params(width) + x.mlp.params(width) + 2 * width * cfg.token_side_dim
            for x in cfg.layers[cfg.loop.start : cfg.loop.stop]
        )
        passed += (cfg.loop.times - 1) * again
    read, pairs_flops = 0, 0.0

    def attended(window):
        """(cached keys in reach, visible query and key pairs)"""
        keys = pairs = 0
        for c, n in lengths:
            first = max(0, c - window + 1)
            keys += c - first
            pairs += sum(min(window, c + k + 1) for k in range(n))
        return keys, pairs

    def add(window, row, per_pair, layers=1):
        nonlocal read, pairs_flops
        keys, pairs = attended(window or 1 << 30)
        read += layers * (keys + tokens) * row  # cached rows read, new rows written
        pairs_flops += 2.0 * layers * pairs * per_pair

    if not runs:
        add(None, 2 * cfg.num_kv_heads * cfg.head_dim, 2 * cfg.num_heads * cfg.head_dim,
            cfg.num_layers)
    for layer in runs:
        m = layer.mixer
        if hasattr(m, "kv_rank"):
            add(m.window, m.kv_rank + m.rot_dim, m.heads * (m.dim + m.rot_dim + m.vdim))
        elif hasattr(m, "softcap"):
            add(m.window, m.kv_heads * (m.dim + m.vdim), m.heads * (m.dim + m.vdim))
        else:  # the delta rule: 7 operations a state element and token, the state written
            pairs_flops += 7.0 * tokens * m.heads * m.dim * m.vdim
            read += 2 * len(lengths) * m.heads * m.dim * m.vdim
    steps = 2 if case["then_decode"] else 1
    bytes_ = steps * (2 * (weights + head) + 4 * logits * vocab) + 2 * read
    flops = 2.0 * tokens * passed + steps * 2.0 * logits * head + pairs_flops
    if steps == 2:
        flops += 2.0 * logits * passed
    return {"bytes": float(bytes_), "flops": float(flops)}


def work(case):
    if case["kind"] == "step":
        return _work_step(case)
    n = case["tokens"]
    if case["kind"] == "sample":
        return {"bytes": 4.0 * n * case["vocab"], "flops": 4.0 * n * case["vocab"]}
    cfg = PRESETS[case["model"]]
    spec = next(x.mlp for x in cfg.layers if hasattr(x.mlp, "experts"))
    E, top, ff, w = spec.experts, spec.top, spec.expert.width, cfg.hidden_size
    touched = E * (1 - (1 - top / E) ** n)
    return {
        "bytes": 2.0 * (touched * 3 * ff * w + n * w + n * top * w + E * w),
        "flops": 2.0 * n * (top * 3 * ff * w + E * w),
    }


def tolerance(case):
    if case["kind"] == "sample":
        # a draw that falls between two sums of the same probabilities
        return {"rel": 0.0, "max": 0.0, "differ": 0.01}
    if case["kind"] == "experts":
        return {"rel": 8e-3, "max": 0.3}
    # 32 layers with a bf16 residual: prompts through another attention kernel differ by
    # 1.5%, largest 0.08; both are 1.6% off the result in 64 bits (fp32 residuals: 0.5 to 1.4%)
    return {"rel": 0.03, "max": 0.3}


# -------------------------------------------------------- the same in 64 bits


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "sample":
        return None
    with torch.no_grad():
        return _EXACT[case.get("model")](state)


def _product(x, w):
    """x @ w^T with w taken to 64 bits in parts."""
    return torch.cat([x @ p.double().t() for p in w.split(1 << 14)], -1)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _softmax_rows(q, k, v, scale, first, window=None, keep=0, cap=None, sink=None):
    """Causal attention of the heads that share k and v: q [Lq, h, d], whose row 0 is at
    position ``first``, over k, v [Lk, d].  Returns [Lq, h, e]."""
    out = []
    for at in range(0, len(q), 1024):
        rows = q[at : at + 1024]
        i = first + at + torch.arange(len(rows), device=q.device).view(-1, 1)
        j = torch.arange(len(k), device=q.device).view(1, -1)
        ok = j <= i
        if window is not None:
            ok &= (i - j < window) | (j < keep)
        s = torch.einsum("qhd,kd->hqk", rows, k) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~ok, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.double().view(-1, 1, 1).expand(-1, len(rows), 1)], -1)
        p = torch.softmax(s, -1)[..., : len(k)]
        out.append(torch.einsum("hqk,ke->qhe", p, v))
    return torch.cat(out)


def _rows_of(state):
    """Per sequence: its rows among the step's tokens, and where they begin in it."""
    at = 0
    for n, (cached, new) in enumerate(state.lengths):
        yield n, slice(at, at + new), cached
        at += new


def _tokens_of(state):
    ids = sum((mine[c : c + n] for mine, (c, n) in zip(state.ids, state.lengths)), [])
    pos = sum((list(range(c, c + n)) for c, n in state.lengths), [])
    last = torch.tensor([r.stop - 1 for _, r, _ in _rows_of(state)], device=DEVICE)
    return (torch.tensor(ids, device=DEVICE),
            torch.tensor(pos, device=DEVICE, dtype=torch.float64), last)


def _angles(pos, n, base):
    a = pos.view(-1, 1) * base ** (-torch.arange(0, n, 2, device=DEVICE, dtype=torch.float64) / n)
    return torch.cos(a).unsqueeze(1), torch.sin(a).unsqueeze(1)


def _exact_llama(state):
    m, cfg = state.engine.model, state.engine.mcfg
    ids, pos, last = _tokens_of(state)
    H, G, d = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    cos, sin = _angles(pos, d, cfg.rope_theta)
    x = m.embed[ids].double()

    def turn(t):
        a, b = t[..., : d // 2], t[..., d // 2 :]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for n, lw in enumerate(m.layers):
        h = _rms(x, cfg.rms_eps) * lw.input_norm.double()
        qkv = _product(h, lw.qkv).view(len(ids), H + 2 * G, d)
        q, k, v = turn(qkv[:, :H]), turn(qkv[:, H : H + G]), qkv[:, H + G :]
        o = torch.empty_like(q)
        for s, rows, cached in _rows_of(state):
            old_k, old_v = state.cached(m.k_caches[n], s), state.cached(m.v_caches[n], s)
            ks, vs = torch.cat([old_k, k[rows]]), torch.cat([old_v, v[rows]])
            if cached and rows.stop - rows.start == 1:  # all heads at once
                w = torch.einsum("gqd,kgd->gqk", q[rows].view(G, H // G, d), ks) * d ** -0.5
                mixed = torch.einsum("gqk,kgd->gqd", torch.softmax(w, -1), vs)
                o[rows] = mixed.reshape(1, H, d)
                continue
            for g in range(G):
                mine = slice(g * (H // G), (g + 1) * (H // G))
                o[rows, mine] = _softmax_rows(
                    q[rows, mine], ks[:, g], vs[:, g], d ** -0.5, cached
                )
        x = x + _product(o.flatten(1), lw.o)
        h = _rms(x, cfg.rms_eps) * lw.post_norm.double()
        parts = []
        for r in h.split(4096):
            gate, up = _product(r, lw.gate_up).chunk(2, -1)
            parts.append(_product(_silu(gate) * up, lw.down))
        x = x + torch.cat(parts)
    h = _rms(x[last], cfg.rms_eps) * m.final_norm.double()
    return [_product(h, m.lm_head)]


def _exact_fetolix(state):
    m, cfg = state.engine.model, state.engine.mcfg
    ids, pos, last = _tokens_of(state)
    W, eps = m.named_tensors(), cfg.rms_eps
    x = x0 = W["embed"][ids].double()

    def layer_norm(t, w):
        return torch.nn.functional.layer_norm(t, t.shape[-1:], w.double(), None, eps)

    def turn(t, base):
        c, s = _angles(pos, t.shape[-1], base)
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)

    for run_, (i, enters) in enumerate(cfg.layer_runs):
        if enters:
            x = _product(torch.cat([x, x0], -1), W["loop.in"])
        p, spec, mlp = f"l{i}.", cfg.layers[i].mixer, cfg.layers[i].mlp
        H, d, r, e, rank = spec.heads, spec.dim, spec.rot_dim, spec.vdim, spec.kv_rank
        h = layer_norm(x, W[p + "norm1"])
        if spec.q_rank:
            low = _rms(_product(h, W[p + "mix.dq"]), eps) * W[p + "mix.dq.norm"].double()
            q = _product(low, W[p + "mix.uq"])
        else:
            q = _product(h, W[p + "mix.q"])
        q = q.view(-1, H, d + r)
        kv = _product(h, W[p + "mix.dkv"])
        latent = _rms(kv[:, :rank], eps) * W[p + "mix.dkv.norm"].double()
        k_rot = turn(kv[:, rank:].unsqueeze(1), spec.rope_base).squeeze(1)
        uk = W[p + "mix.uk"].double().view(H, d, rank)
        uv = W[p + "mix.uv"].double().view(H, e, rank)
        # queries and results in terms of the latents
        q = torch.cat([torch.einsum("nhd,hdr->nhr", q[..., :d], uk),
                       turn(q[..., d:], spec.rope_base)], -1)
        o = q.new_empty(len(ids), H, rank)
        for s, rows, cached in _rows_of(state):
            keys = torch.cat([state.cached(m.caches[run_], s),
                              torch.cat([latent[rows], k_rot[rows]], -1)])
            o[rows] = _softmax_rows(q[rows], keys, keys[:, :rank], spec.scale, cached,
                                    spec.window)
        o = torch.einsum("nhr,her->nhe", o, uv)
        o = o * torch.sigmoid(_product(h, W[p + "mix.g"])).unsqueeze(-1)
        y = _product(o.flatten(1), W[p + "mix.o"])
        gate = _product(h, W[p + "mlp.gate"]).clamp(max=mlp.limit)
        up = _product(h, W[p + "mlp.up"]).clamp(-mlp.limit, mlp.limit)
        act = gate * torch.sigmoid(mlp.alpha * gate) * (up + mlp.offset)
        x = x + y + _product(act, W[p + "mlp.down"])
        side = W["side.embed"][ids][:, i * cfg.token_side_dim : (i + 1) * cfg.token_side_dim]
        z = torch.nn.functional.gelu(_product(x, W[p + "side.gate"]), approximate="tanh")
        y = _rms(_product(z * side.double(), W[p + "side.proj"]), eps)
        x = x + y * W[p + "side.norm"].double()
    return [_product(layer_norm(x[last], W["final.norm"]), W["embed"])]


def _exact_delta_heads(h, W, p, spec, eps):
    """One sequence's rows through a delta layer, ahead of its output projection."""
    T, H, G, D, V = len(h), spec.heads, spec.kv_heads, spec.dim, spec.vdim

    def conv(name, heads, size):
        x, w = _product(h, W[p + name]), W[p + name + ".conv"].double()
        taps = w.shape[1]
        x = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
        return _silu(sum(x[n : n + T] * w[:, n] for n in range(taps))).view(T, heads, size)

    def unit(t):
        return t / torch.sqrt((t * t).sum(-1, keepdim=True) + spec.unit_eps)

    q, k = unit(conv("q", G, D)) * D ** -0.5, unit(conv("k", G, D))
    q, k = (t.repeat_interleave(H // G, 1) for t in (q, k))
    v, beta = conv("v", H, V), torch.sigmoid(_product(h, W[p + "b"]))
    z = _product(_product(h, W[p + "a1"]), W[p + "a2"]) + W[p + "dt_bias"].double()
    rate = torch.exp(W[p + "A_log"].double()).view(1, H, 1)
    decay = torch.exp(-rate * torch.nn.functional.softplus(z.view(T, H, D), threshold=40))
    gate = torch.sigmoid(_product(_product(h, W[p + "g1"]), W[p + "g2"])).view(T, H, V)
    S, out = h.new_zeros(H, D, V), h.new_empty(T, H, V)
    for t in range(T):
        S *= decay[t].unsqueeze(2)
        u = beta[t].view(H, 1, 1) * (v[t].unsqueeze(1) - k[t].unsqueeze(1) @ S)
        S.baddbmm_(k[t].unsqueeze(2), u)
        out[t] = (q[t].unsqueeze(1) @ S).squeeze(1)
    return (_rms(out, eps) * W[p + "norm"].double() * gate).flatten(1)


def _exact_tezinex(state):
    m, cfg = state.engine.model, state.engine.mcfg
    W, eps, width = m.named_tensors(), cfg.rms_eps, cfg.hidden_size
    firsts, seconds = [], []
    for mine in state.ids:
        T = len(mine)
        a = torch.arange(T, device=DEVICE, dtype=torch.float64).view(-1, 1)
        c = torch.arange(width, device=DEVICE)
        a = a * cfg.position_base ** (-2.0 * (c // 2).double() / width)
        x = W["embed"][torch.tensor(mine, device=DEVICE)].double()
        x = x + torch.where(c % 2 == 1, torch.cos(a), torch.sin(a))
        states, kv = [x], {}

        def norm(t, name):
            return _rms(t, eps) * (1 + W[name].double())

        for i, layer in enumerate(cfg.layers):
            p, spec = f"l{i}.mix.", layer.mixer
            h = norm(x, f"l{i}.norm1")
            if not hasattr(spec, "softcap"):
                y = _exact_delta_heads(h, W, p, spec, eps)
            else:
                H, G = spec.heads, spec.kv_heads

                def rows(name, heads):
                    t = _product(h, W[p + name]) + W[p + name + ".b"].double()
                    return t.view(T, heads, -1)

                if spec.kv_from is None:
                    kv[i] = rows("k", G), rows("v", G)
                k, v = kv[i if spec.kv_from is None else spec.kv_from]
                q, per = rows("q", H), H // G
                y = torch.cat([
                    _softmax_rows(
                        q[:, g * per : (g + 1) * per], k[:, g], v[:, g], spec.scale, 0,
                        spec.window, spec.keep_first, spec.softcap,
                        W[p + "sink"][g * per : (g + 1) * per],
                    ) for g in range(G)
                ], 1).flatten(1)
            x = x + cfg.residual_mult * norm(_product(y, W[p + "o"]), f"l{i}.norm1b")
            h, q = norm(x, f"l{i}.norm2"), f"l{i}.mlp."
            y = _silu(_product(h, W[q + "gate"])) * _product(h, W[q + "up"])
            x = x + cfg.residual_mult * norm(_product(y, W[q + "down"]), f"l{i}.norm2b")
            states.append(x)
            x = sum(c * s for c, s in zip(W[f"l{i}.dwa"].double(), states))
        x = norm(x[-2:], "final.norm")
        logits = _product(x, W["embed"])
        logits = cfg.logit_softcap * torch.tanh(logits / cfg.logit_softcap)
        firsts.append(logits[0])
        seconds.append(logits[1])
    return [torch.stack(firsts), torch.stack(seconds)]


def _exact_experts(state):
    spec, layer, h = state.spec, state.layer, state.h.double()
    W = layer.export("")
    z = _product(h, W["router"])
    if layer.router_bias is not None:
        z = z + layer.router_bias.double()
    top, ids = torch.topk(z, spec.top, -1)
    rows = h.new_empty(len(h), spec.top, state.width)
    glu = spec.expert
    for e in range(spec.experts):
        n, j = torch.nonzero(ids == e, as_tuple=True)
        gate = _product(h[n], W[f"e{e}.gate"]).clamp(max=glu.limit)
        up = _product(h[n], W[f"e{e}.up"]).clamp(-glu.limit, glu.limit)
        act = gate * torch.sigmoid(glu.alpha * gate) * (up + glu.offset)
        rows[n, j] = _product(act, W[f"e{e}.down"])
    return rows, torch.softmax(top, -1)


_EXACT = {
    "llama3-8b": _exact_llama, "llama2-7b": _exact_llama, "fetolix-2b": _exact_fetolix,
    "tezinex-2b": _exact_tezinex, "lobuvik-8b": _exact_experts, "lobuvik-2b": _exact_experts,
}
