"""GPU numerics: every CDNA4 kernel against its plain-PyTorch fp32 reference
(SURVEY.md §4 implication: kernel-level golden tests are a new test tier).

All tests are @gpu — run via gpurun on an MI355X.
"""
import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

from agentcontrolplane_amd import ops
from agentcontrolplane_amd.ops import reference as ref

requires_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs MI355X")


def hip():
    from agentcontrolplane_amd.ops import hip as m

    return m


def maxerr(a, b):
    return (a.float() - b.float()).abs().max().item()


def assert_one_ulp(got, want):
    """bf16 results may round to neighbours: 2^-7 of the value, of one if it is smaller."""
    err = (got.float() - want.float()).abs() / want.float().abs().clamp(min=1.0)
    assert err.max().item() <= 2.0 ** -7


@requires_gpu
@pytest.mark.parametrize("n,h", [(1, 4096), (17, 4096), (256, 8192), (33, 256)])
def test_rmsnorm(n, h):
    x = torch.randn(n, h, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(h, dtype=torch.bfloat16, device="cuda").abs() + 0.5
    out = hip().rmsnorm(x, w, 1e-5)
    want = ref.rmsnorm(x.cpu(), w.cpu(), 1e-5)
    assert_one_ulp(out.cpu(), want)


@requires_gpu
def test_fused_add_rmsnorm():
    n, h = 64, 4096
    x = torch.randn(n, h, dtype=torch.bfloat16, device="cuda")
    r = torch.randn(n, h, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(h, dtype=torch.bfloat16, device="cuda").abs() + 0.5
    xc, rc = x.cpu().clone(), r.cpu().clone()
    out, new_r = hip().fused_add_rmsnorm(x, r, w, 1e-5)
    want_out, want_r = ref.fused_add_rmsnorm(xc, rc, w.cpu(), 1e-5)
    assert maxerr(new_r.cpu(), want_r) < 0.05
    assert_one_ulp(out.cpu(), want_out)


@requires_gpu
@pytest.mark.parametrize("n,inter", [(4, 14336), (129, 512)])
def test_swiglu(n, inter):
    gu = torch.randn(n, 2 * inter, dtype=torch.bfloat16, device="cuda")
    out = hip().swiglu(gu)
    want = ref.swiglu(gu.cpu())
    assert_one_ulp(out.cpu(), want)


def _make_cache(num_blocks, bs, hkv, d, device, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn(num_blocks, bs, hkv, d, generator=g, dtype=torch.float32).to(dtype)
    v = torch.randn(num_blocks, bs, hkv, d, generator=g, dtype=torch.float32).to(dtype)
    return k.to(device), v.to(device)


@requires_gpu
def test_rope_cache():
    N, Hq, Hkv, D, P = 37, 4, 2, 128, 512
    torch.manual_seed(0)
    q = torch.randn(N, Hq, D, dtype=torch.bfloat16, device="cuda")
    k = torch.randn(N, Hkv, D, dtype=torch.bfloat16, device="cuda")
    v = torch.randn(N, Hkv, D, dtype=torch.bfloat16, device="cuda")
    kc, vc = _make_cache(16, 16, Hkv, D, "cuda")
    kc.zero_(); vc.zero_()
    pos = torch.randint(0, P, (N,), device="cuda", dtype=torch.long)
    slots = torch.randperm(16 * 16, device="cuda")[:N].long()
    cos_sin = ref.build_cos_sin(P, D, 500000.0, "cuda")
    qc, kcpu, vcpu = q.cpu().clone(), k.cpu().clone(), v.cpu().clone()
    kc_cpu = torch.zeros(16, 16, Hkv, D, dtype=torch.bfloat16)
    vc_cpu = torch.zeros_like(kc_cpu)
    q2, k2 = hip().rope_and_cache(q, k, v, pos, slots, kc, vc, cos_sin)
    ref.rope_and_cache(
        qc, kcpu, vcpu, pos.cpu(), slots.cpu(), kc_cpu, vc_cpu, cos_sin.cpu()
    )
    assert maxerr(q2.cpu(), qc) < 0.03
    assert maxerr(k2.cpu(), kcpu) < 0.03
    assert maxerr(kc.cpu(), kc_cpu) < 0.03
    assert maxerr(vc.cpu(), vc_cpu) < 0.03


@requires_gpu
@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_decode_attn(G):
    torch.manual_seed(1)
    B, Hkv, D, bs = 5, 2, 128, 16
    Hq = Hkv * G
    num_blocks = 64
    kc, vc = _make_cache(num_blocks, bs, Hkv, D, "cuda")
    seq_lens = torch.tensor([1, 17, 63, 200, 333], dtype=torch.long)
    max_blocks = int((seq_lens.max() + bs - 1) // bs)
    # random non-overlapping block tables
    perm = torch.randperm(num_blocks)
    tables = torch.zeros(B, max_blocks, dtype=torch.long)
    off = 0
    for i in range(B):
        nb = int((seq_lens[i] + bs - 1) // bs)
        tables[i, :nb] = perm[off : off + nb]
        off += nb
    q = torch.randn(B, Hq, D, dtype=torch.bfloat16, device="cuda")
    scale = 1.0 / math.sqrt(D)
    out = hip().attention_decode_raw(
        q, kc, vc, tables.to("cuda"), seq_lens.to("cuda"), scale
    )
    want = ref.attention_decode_raw(
        q.cpu().float(), kc.cpu().float(), vc.cpu().float(), tables, seq_lens, scale
    )
    assert maxerr(out.cpu(), want) < 0.03


@requires_gpu
@pytest.mark.parametrize("block", [8, 16, 24, 64])
@pytest.mark.parametrize("H,G", [(8, 8), (7, 1), (6, 2), (16, 2)])
@pytest.mark.parametrize("lens", [
    [1], [32, 0, 33], [31, 64, 65, 700, 128, 129, 1, 3000], [40, 7] * 70, [100] * 3 + [5] * 1100,
], ids=["one", "none", "ragged", "over_64", "whole"])
def test_decode_pieces(block, H, G, lens):
    """Steps cut into pieces and merged, or with whole sequences; what no token has written
    is NaN."""
    torch.manual_seed(len(lens))
    need = [-(-n // block) for n in lens]
    order = torch.randperm(sum(need) + 1)
    tables = torch.zeros(len(lens), max(need) + 2, dtype=torch.int32)
    kc = torch.full((len(order), block, G, 128), float("nan"), device="cuda").bfloat16()
    vc, at, rows = kc.clone(), 0, []
    for b, (n, k) in enumerate(zip(lens, need)):
        tables[b, :k] = order[at : at + k]
        p = torch.arange(n)
        rows.append(order[at : at + k][p // block] * block + p % block)
        at += k
    slots = torch.cat(rows).cuda()
    for c in (kc, vc):
        c.view(-1, G, 128)[slots] = torch.randn(len(slots), G, 128, device="cuda").bfloat16()
    q = torch.randn(len(lens), H, 128, device="cuda").bfloat16()
    out = hip().attention_decode_raw(
        q, kc, vc, tables.cuda(), torch.tensor(lens).cuda(), 0.09
    ).float()
    keys, values = (c.view(-1, G, 128).float() for c in (kc, vc))
    for b in {*range(min(10, len(lens))), len(lens) - 1}:
        k, v = (c[rows[b].cuda()].repeat_interleave(H // G, 1) for c in (keys, values))
        w = torch.softmax((k * q[b].float()).sum(-1) * 0.09, 0)
        # fp32 but for the result: 2^-9 of values up to 5
        assert maxerr(out[b], (w.unsqueeze(-1) * v).sum(0)) < 0.012, (b, lens[b])


@requires_gpu
@pytest.mark.parametrize("step", ["prompt", "decode"])
def test_attention_writes_into_any_contiguous_memory(step):
    """``out`` off a 16-byte boundary, flat, or larger than the result; strided ones are refused."""
    from op_helpers import make_batch

    H, G, n = 8, 2, 37
    torch.manual_seed(1)
    batch, _, tables, pages = make_batch([(0, n)] if step == "prompt" else [(n, 1)] * 3, 16, "cuda")
    kc, vc = torch.randn(2, pages, 16, G, 128, device="cuda").bfloat16()
    rows = n if step == "prompt" else 3
    q = torch.randn(rows, H, 128, device="cuda").bfloat16()
    attend = hip().attention_prefill_batch if step == "prompt" else hip().attention_decode_batch
    want = attend(q, kc, vc, batch, 0.1).flatten()
    size = rows * H * 128
    for shift, more in [(0, 0), (3, 0), (3, 5), (8, 17)]:
        space = torch.full((size + 64,), 7.0, device="cuda").bfloat16()
        out = space[shift : shift + size + more]
        if more == 0:
            out = out.view(rows, H * 128)
        assert attend(q, kc, vc, batch, 0.1, out=out) is out
        assert torch.equal(space[shift : shift + size], want)
        assert (space[:shift] == 7).all() and (space[shift + size :] == 7).all()
    with pytest.raises(RuntimeError, match="contiguous"):
        attend(q, kc, vc, batch, 0.1, out=q.new_empty(rows, H, 256)[..., :128])


STEADY = {  # lengths, heads, key heads, head size, options
    "ragged": ([300 + 97 * i * 53 % 3701 for i in range(44)], 32, 8, 128, {}),
    "over_64": ([150 + 97 * i * 61 % 1501 for i in range(90)], 16, 8, 128, {}),
    "one": ([4003], 28, 4, 128, {}),
    "whole": ([301 + 97 * i * 37 % 403 for i in range(130)], 16, 8, 128, {}),
    "window": ([200 + 97 * i * 71 % 2801 for i in range(41)], 16, 8, 128,
               dict(window=1000, keep_first=5, cap=20.0, sink=True)),
    "sigmoid": ([900 + 97 * i * 71 % 1801 for i in range(24)], 12, 4, 128, dict(sigmoid=True)),
    "wide": ([700 + 97 * i * 31 % 2301 for i in range(20)], 12, 2, 256,
             dict(window=1500, keep_first=70, sink=True)),
    "narrow": ([500 + 97 * i * 31 % 2301 for i in range(33)], 12, 4, 64, dict(window=1 << 20)),
}


@requires_gpu
@pytest.mark.parametrize("block", [16, 24, 64])
@pytest.mark.parametrize("case", STEADY)
def test_decode_over_many_blocks(case, block):
    """Several blocks of 32 keys a wave, in pieces of one size, of sizes that are evened out and
    in whole sequences; what no token has written is NaN."""
    lens, H, G, d, options = STEADY[case]
    options = dict(options)
    gen = torch.Generator().manual_seed(len(lens))
    need = [-(-n // block) for n in lens]
    order = torch.randperm(sum(need) + 1, generator=gen)
    tables = torch.zeros(len(lens), max(need) + 3, dtype=torch.int32)
    kc, vc = torch.full((2, len(order), block, G, d), float("nan"), device="cuda").bfloat16()
    rows, at = [], 0
    for b, (n, k) in enumerate(zip(lens, need)):
        tables[b, :k] = order[at : at + k]
        p = torch.arange(n)
        rows.append((order[at : at + k][p // block] * block + p % block).cuda())
        at += k
        for c in (kc, vc):
            c.view(-1, G, d)[rows[b]] = torch.randn(n, G, d, device="cuda").bfloat16()
    q = (2 * torch.randn(len(lens), H, d, generator=gen)).bfloat16().cuda()
    seq_lens, scale = torch.tensor(lens, dtype=torch.int32).cuda(), d ** -0.5
    sink = torch.randn(H, generator=gen).cuda() if options.pop("sink", None) else None
    if options:
        batch = SimpleNamespace(
            num_prefill_tokens=0, prefills=[], num_decode=len(lens),
            decode_tables_i32=lambda t=tables.cuda(): t, decode_lens_i32=lambda: seq_lens,
        )
        form = {"cap": None, "window": None, "keep_first": 0, **options}
        out = torch.empty_like(q)
        hip().grouped_attention(q, kc, vc, batch, scale, sink=sink, out=out, **form)
    else:
        form = {"cap": None, "window": None, "keep_first": 0}
        out = hip().attention_decode_raw(q, kc, vc, tables.cuda(), seq_lens, scale)
    for b, n in enumerate(lens):
        k, v = (c.view(-1, G, d)[rows[b]].float().repeat_interleave(H // G, 1) for c in (kc, vc))
        s = (k * q[b].float()).sum(-1) * scale
        if form["cap"]:
            s = form["cap"] * torch.tanh(s / form["cap"])
        if form["window"]:
            p = torch.arange(n, device="cuda")[:, None]
            s = s.masked_fill((p <= n - 1 - form["window"]) & (p >= form["keep_first"]), -math.inf)
        if form.get("sigmoid"):
            w = torch.sigmoid(s)
        else:
            w = torch.softmax(s if sink is None else torch.cat([s, sink[None]]), 0)[:n]
        want = (w.unsqueeze(-1) * v).sum(0)
        # fp32 but for the result: 2^-9 of it, and 2^-20 of sums of up to 4003 terms
        slack = 2.0 ** -8 * want.abs() + 2.0 ** -20 * (w.unsqueeze(-1) * v.abs()).sum(0) + 1e-4
        assert ((out[b].float() - want).abs() <= slack).all(), (b, n)


@requires_gpu
def test_decode_pieces_of_wide_tables():
    """Room for 2^22 blocks of 32 keys, whose count is divided in another way: the same pieces."""
    torch.manual_seed(2)
    lens = torch.tensor([700, 33, 2100, 0, 1, 4000, 950], dtype=torch.int32).cuda()
    tables = torch.randint(0, 90, (7, 260), dtype=torch.int32).cuda()
    kc, vc = torch.randn(2, 90, 16, 4, 128, device="cuda").bfloat16()
    q = torch.randn(7, 16, 128, device="cuda").bfloat16()
    wide = torch.zeros(7, 1 << 21, dtype=torch.int32, device="cuda")
    wide[:, :260] = tables
    got, want = (hip().attention_decode_raw(q, kc, vc, t, lens, 0.1) for t in (wide, tables))
    assert torch.equal(got, want)


@requires_gpu
def test_mfma_fragment_layout_probe():
    """The assumed A/B/D lane maps for v_mfma_f32_32x32x16_bf16 must
    reproduce a plain matmul (asymmetric operands per guide G9/rule 16)."""
    import torch

    from agentcontrolplane_amd import _C

    torch.manual_seed(7)
    a = (torch.randn(32, 16) * 0.5).bfloat16().cuda()
    b = (torch.randn(16, 32) * 0.5).bfloat16().cuda()
    d = _C.mfma_probe(a, b)
    want = a.cpu().float() @ b.cpu().float()
    err = (d.cpu() - want).abs().max().item()
    assert err < 0.05, f"fragment layout mismatch: max err {err}"


@requires_gpu
@pytest.mark.parametrize("impl", ["v0", "mfma"])
def test_prefill_attn_multi_seq(impl, monkeypatch):
    """Three chunks with different ctx offsets in one batched launch."""
    from agentcontrolplane_amd.engine.batch import FlatBatch, SeqMeta
    from agentcontrolplane_amd.ops import hip as hip_mod

    monkeypatch.setattr(hip_mod, "_PREFILL_IMPL", impl)
    torch.manual_seed(2)
    Hq, Hkv, D, bs = 4, 2, 128, 16
    num_blocks = 128
    kc, vc = _make_cache(num_blocks, bs, Hkv, D, "cuda")
    # (query_len, ctx_len)
    shapes = [(70, 0), (1, 129), (65, 63)]
    perm = torch.randperm(num_blocks)
    metas = []
    off = 0
    rows = 0
    for qlen, ctx in shapes:
        S = qlen + ctx
        nb = (S + bs - 1) // bs
        metas.append(
            SeqMeta(
                seq_id=0, query_len=qlen, seq_len=S, ctx_len=ctx,
                block_table=perm[off : off + nb].tolist(), needs_logits=True,
            )
        )
        off += nb
        rows += qlen
    dummy = torch.empty(0)
    batch = FlatBatch(
        token_ids=torch.empty(rows, device="cuda"), positions=dummy,
        slot_mapping=dummy, prefills=metas, num_prefill_tokens=rows,
        decode_seq_ids=[], decode_block_tables=None, decode_seq_lens=None,
        logit_rows=dummy, sample_seq_ids=[],
    )
    q = torch.randn(rows, Hq, D, dtype=torch.bfloat16, device="cuda")
    scale = 1.0 / math.sqrt(D)
    out = hip().attention_prefill_batch(q, kc, vc, batch, scale)
    # oracle per sequence on fp32 CPU
    row = 0
    for m in metas:
        want = ref.attention_prefill(
            q[row : row + m.query_len].cpu().float(), kc.cpu().float(),
            vc.cpu().float(), m.block_table, m.seq_len, m.ctx_len, scale,
        )
        err = maxerr(out[row : row + m.query_len].cpu(), want)
        assert err < 0.03, f"chunk {m}: err {err}"
        row += m.query_len


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [513, 1023, 16385, 50257, 128256, 262144])
def test_fullvocab_draws_lie_in_the_kept_cdf(V, dtype):
    """Rows of every kind: spread, alike, in two values, with steps far below the largest, with
    -inf, with masks; the drawn token's part of the 64-bit CDF holds the uniform."""
    torch.manual_seed(V)
    rows = [
        torch.randn(V) * 2.5, torch.full((V,), 1.5), torch.randint(0, 2, (V,)).float(),
        torch.randn(V) * 1e-6, torch.randn(V) * 1e4, torch.randn(V) * 3,
        torch.where(torch.arange(V) % 3 == 0, torch.randn(V), torch.tensor(-float("inf"))),
        torch.cat([torch.tensor([40.0]), torch.randn(V - 1)]),
    ]
    kinds = [(0, 1.0), (1, 1.0), (50, 1.0), (5000, 1.0), (0, 0.9), (0, 0.999), (40, 0.5)]
    x = torch.stack(rows).to(dtype).cuda()
    mask = torch.rand(2, V) < 0.02
    mask[1] = False
    mask[1, V - 1] = True
    for k, p in kinds:
        for mapped in (None, [0, 1, -1, 0, 1, 0, 0, -1]):
            u = torch.rand(len(rows))
            got = hip().softmax_sample(
                x, torch.full((len(rows),), 0.8).cuda(),
                torch.full((len(rows),), k).cuda(), torch.full((len(rows),), p).cuda(), None,
                mask.cuda() if mapped else None, u.cuda(),
                torch.tensor(mapped, dtype=torch.int32).cuda() if mapped else None,
            ).tolist()
            for r in range(len(rows)):
                v = x[r].double().cpu()
                if mapped and mapped[r] >= 0:
                    v = v.masked_fill(~mask[mapped[r]], -float("inf"))
                w = torch.exp((v - v.max()) / 0.8)
                order = torch.sort(v, descending=True).values
                if 0 < k < V:
                    w[v < order[k - 1]] = 0
                at = v[got[r]]
                if p < 1:  # the weight of what is larger is within p of the kept
                    assert w[v > at].sum() <= (p + 1e-5) * w.sum(), (r, k, p)
                    above = torch.cumsum(torch.exp((order - order[0]) / 0.8), 0)
                    edge = order[int((above >= p * w.sum()).nonzero()[0])]
                    w[v < edge] = 0
                    if at < edge:  # a boundary within rounding
                        continue
                c = torch.cumsum(w, 0) / w.sum()
                lo = c[got[r] - 1].item() if got[r] else 0.0
                # sums of 262144 weights in fp32, in 256 parts: 2^-24 * (1024 + 256)
                assert lo - 1e-4 <= u[r] <= c[got[r]].item() + 1e-4, (r, k, p)


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [4093, 4096, 4097, 8191, 8192, 8193])
def test_fullvocab_draws_with_few_and_many_threads(V, dtype):
    """Around the sizes up to which a row has 256 threads, with few rows and with many: the
    same tokens, and stripes of 16, 17 and 32 tokens."""
    test_fullvocab_draws_lie_in_the_kept_cdf(V, dtype)
    n = 300
    x = (2.5 * torch.randn(n, V)).to(dtype).cuda()
    args = [torch.full((n,), 0.8).cuda(), torch.tensor([0, 40, 0] * 100).cuda(),
            torch.tensor([1.0, 1.0, 0.9] * 100).cuda()]
    u = torch.rand(n).cuda()
    many = hip().softmax_sample(x, *args, None, None, u)
    few = torch.cat([
        hip().softmax_sample(x[i : i + 100], *(a[i : i + 100] for a in args), None, None,
                             u[i : i + 100]) for i in range(0, n, 100)
    ])
    assert torch.equal(many, few)


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [700, 50257])
@pytest.mark.parametrize("T,k,p", [(0.0, 0, 1.0), (0.8, 0, 1.0), (0.8, 1, 1.0), (0.8, 5, 1.0),
                                   (0.8, 0, 0.9), (0.8, 40, 0.5)])
def test_fullvocab_rows_with_infinities_and_nan(V, dtype, T, k, p):
    """Tokens are allowed ones, an infinite logit wins where the largest must, a masked one and
    other rows' change nothing."""
    torch.manual_seed(V)
    x = torch.randn(8, V)
    x[1, 3] = math.inf
    x[2, [5, V // 2, V - 2]] = math.inf
    x[3, [0, 9, V - 1]] = math.nan
    x[4, 11] = math.nan  # masked
    x[5, 12] = math.inf  # masked
    x[6, 13] = math.inf
    x[6, 14] = -math.nan
    mask = torch.rand(2, V) < 0.3
    mask[:, [11, 12]] = False
    mask[1, 20] = True
    rows = [-1, -1, -1, -1, 0, 1, -1, 1]
    u = torch.rand(8)

    def draw(x):
        n = len(x)
        return hip().softmax_sample(
            x.to(dtype).cuda(), torch.full((n,), T).cuda(), torch.full((n,), k).cuda(),
            torch.full((n,), p).cuda(), None, mask.cuda(), u.cuda(),
            torch.tensor(rows, dtype=torch.int32).cuda(),
        ).tolist()

    got = draw(x)
    for r, m in enumerate(rows):
        assert 0 <= got[r] < V and (m < 0 or mask[m, got[r]]), r
    if T == 0:
        assert got[1] == 3 and got[2] == 5 and got[6] == 13
    if k == 1:
        assert got[1] == 3 and got[2] in (5, V // 2, V - 2)
    finite = torch.where(x.isfinite(), x, torch.zeros(()))
    plain = draw(finite)
    assert [got[r] for r in (0, 4, 5, 7)] == [plain[r] for r in (0, 4, 5, 7)]


@requires_gpu
@pytest.mark.parametrize("k", [0, 3])
@pytest.mark.parametrize("p", [0.0, -1.0])
@pytest.mark.parametrize("V", [600, 128256])
def test_fullvocab_top_p_of_zero_keeps_the_largest(V, p, k):
    """The nucleus always has the largest allowed logits, as many as are equal, as in the oracle; a
    negative p is taken for zero."""
    torch.manual_seed(V)
    x = torch.randn(6, V)
    x[1, [7, V // 2, V - 3]] = 9.0
    x[2, 0] = 50.0
    x[3] = -2.0
    x[4, : V // 2] = -math.inf
    mask = torch.rand(2, V) < 0.05
    mask[:, 0] = False
    rows = [-1, -1, 0, -1, 1, 1]
    u = torch.tensor([0.5, 0.5, 0.1, 0.999, 0.3, 0.0])
    got = hip().softmax_sample(
        x.cuda(), torch.full((6,), 0.7).cuda(), torch.full((6,), k).cuda(),
        torch.full((6,), p).cuda(), None, mask.cuda(), u.cuda(),
        torch.tensor(rows, dtype=torch.int32).cuda(),
    ).tolist()
    for r, m in enumerate(rows):
        v = x[r] if m < 0 else x[r].masked_fill(~mask[m], -math.inf)
        largest = (v == v.max()).nonzero()[:, 0].tolist()
        assert got[r] == largest[int(u[r].double().item() * len(largest))], r


@requires_gpu
@pytest.mark.parametrize("block", [8, 16, 24, 64])
@pytest.mark.parametrize("H,G,scale", [(8, 8, 0.09), (6, 2, -0.09), (4, 1, 0.0)])
def test_prompt_tiles_over_pages(block, H, G, scale):
    """Chunks that end in, at and past tiles of 64 keys and 128 rows, on pages of every
    kind; what no token has written is NaN."""
    from op_helpers import make_batch

    chunks = [(0, 1), (0, 63), (5, 59), (0, 129), (300, 5), (127, 130)]
    batch, _, tables, pages = make_batch(chunks, block, "cuda")
    kc = torch.full((pages, block, G, 128), float("nan"), device="cuda").bfloat16()
    vc = kc.clone()
    for m in batch.prefills:
        slots = [m.block_table[p // block] * block + p % block for p in range(m.seq_len)]
        for c in (kc, vc):
            c.view(-1, G, 128)[slots] = torch.randn(m.seq_len, G, 128, device="cuda").bfloat16()
    rows = batch.num_prefill_tokens
    q = torch.randn(rows, (H + 3) * 128, device="cuda").bfloat16()
    q = q.as_strided((rows, H, 128), (q.stride(0), 128, 1), 8)
    out = hip().attention_prefill_batch(q, kc, vc, batch, scale)
    row = 0
    for m in batch.prefills:
        mine = slice(row, row + m.query_len)
        want = ref.attention_prefill(
            q[mine].cpu().float(), kc.cpu().float(), vc.cpu().float(), m.block_table,
            m.seq_len, m.ctx_len, scale,
        )
        # weights and results are rounded to 8 bits: 2 * 2^-9 of values up to 5
        assert maxerr(out[mine].cpu(), want) < 0.02, m
        row += m.query_len


@requires_gpu
@pytest.mark.parametrize("block", [16, 24, 64])
@pytest.mark.parametrize("d,v", [(64, 256), (256, 64), (256, 128), (256, 256)])
@pytest.mark.parametrize("form", [dict(window=90, keep_first=3, sink=True), dict(sigmoid=True)])
def test_prompt_head_sizes_over_pages(block, d, v, form):
    """Every count of keys that one load brings, on pages of every kind; what no token has
    written is NaN."""
    from op_helpers import make_batch

    H, G, scale = 6, 2, d ** -0.5
    form = {"cap": None, "window": None, "keep_first": 0, **form}
    gen = torch.Generator().manual_seed(d + v)
    batch, _, _, pages = make_batch([(0, 131), (70, 65), (250, 7)], block, "cuda")
    kc = torch.full((pages, block, G, d), float("nan"), device="cuda").bfloat16()
    vc = torch.full((pages, block, G, v), float("nan"), device="cuda").bfloat16()
    q = torch.randn(batch.num_prefill_tokens, H, d, generator=gen).bfloat16().cuda()
    sink = torch.randn(H, generator=gen).cuda() if form.pop("sink", None) else None
    slots = []
    for m in batch.prefills:
        p = torch.arange(m.seq_len)
        slots.append((torch.tensor(m.block_table)[p // block] * block + p % block).cuda())
        for c in (kc, vc):
            c.view(-1, G, c.shape[3])[slots[-1]] = torch.randn(
                m.seq_len, G, c.shape[3], generator=gen).bfloat16().cuda()
    out = torch.empty(len(q), H, v, dtype=torch.bfloat16, device="cuda")
    hip().grouped_attention(q, kc, vc, batch, scale, sink=sink, out=out, **form)
    row = 0
    for m, at in zip(batch.prefills, slots):
        mine = slice(row, row + m.query_len)
        row += m.query_len
        k, x = (c.view(-1, G, c.shape[3])[at].float().repeat_interleave(H // G, 1)
                for c in (kc, vc))
        s = (q[mine].float()[:, None] * k).sum(-1) * scale  # [queries, keys, H]
        pos = m.ctx_len + torch.arange(m.query_len, device="cuda")[:, None, None]
        key = torch.arange(m.seq_len, device="cuda")[None, :, None]
        hidden = key > pos
        if form["window"]:
            hidden |= (key <= pos - form["window"]) & (key >= form["keep_first"])
        s = s.masked_fill(hidden, -math.inf)
        if form.get("sigmoid"):
            w = torch.sigmoid(s)
        else:
            w = torch.softmax(torch.cat([s, sink.expand(len(s), 1, H)], 1), 1)[:, :-1]
        want = torch.einsum("nkh,khv->nhv", w, x)
        # each weight is rounded to 8 bits, and the result
        slack = 2.0 ** -8 * (torch.einsum("nkh,khv->nhv", w, x.abs()) + want.abs()) + 1e-3
        assert ((out[mine].float() - want).abs() <= slack).all(), m


@requires_gpu
@pytest.mark.parametrize("spread", [1.0, 4.0])
def test_prompt_error_against_64_bits(spread):
    """Weights rounded to 16 bits make most of the error, and all of it above the result's own
    rounding: it is no larger than that of a softmax over tiles of 32 keys whose denominator has
    the weights before rounding."""
    from op_helpers import make_batch

    n, H, scale = 900, 16, 128 ** -0.5
    gen = torch.Generator().manual_seed(1)
    batch, _, _, pages = make_batch([(0, n)], 16, "cuda")
    table = torch.tensor(batch.prefills[0].block_table)
    slots = table[torch.arange(n) // 16] * 16 + torch.arange(n) % 16
    q, k, v = (torch.randn(n, H, 128, generator=gen).mul(x).bfloat16() for x in (spread, 1, 1))
    kc, vc = torch.zeros(2, pages * 16, H, 128, dtype=torch.bfloat16)
    kc[slots], vc[slots] = k, v
    got = hip().attention_prefill_batch(
        q.cuda(), *(c.view(pages, 16, H, 128).cuda() for c in (kc, vc)), batch, scale
    ).cpu().double()
    hidden = torch.ones(n, n).triu(1).bool()
    err = tiles = 0.0
    for h in range(H):
        s = (q[:, h].float() @ k[:, h].float().T * scale).masked_fill(hidden, -math.inf)
        values = v[:, h].double()
        want = torch.softmax(s.double(), -1) @ values
        top, o, total = torch.full((n, 1), -1e30), 0.0, 0.0
        for t in range(0, n, 32):
            up = torch.maximum(top, s[:, t : t + 32].amax(1, keepdim=True))
            w = torch.exp(s[:, t : t + 32] - up)
            down = torch.exp(top - up).double()
            o = o * down + w.bfloat16().double() @ values[t : t + 32]
            total = total * down + w.double().sum(1, keepdim=True)
            top = up
        tiles += ((o / total).bfloat16().double() - want).pow(2).sum().item()
        err += (got[:, h] - want).pow(2).sum().item()
    assert err <= tiles, (err / tiles) ** 0.5


@requires_gpu
def test_sample_greedy_and_filters():
    torch.manual_seed(3)
    B, V = 64, 261
    logits = torch.randn(B, V, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(0)
    zeros = torch.zeros(B, device="cuda")
    ones = torch.ones(B, device="cuda")
    offk = torch.zeros(B, dtype=torch.long, device="cuda")
    # greedy == argmax
    out = hip().softmax_sample(logits, zeros, offk, ones, gen)
    assert torch.equal(out, logits.argmax(-1))
    # top-k: sampled ids within the row's top-k set
    k = 5
    out = hip().softmax_sample(logits, ones, torch.full_like(offk, k), ones, gen)
    topk = logits.topk(k, dim=-1).indices
    for i in range(B):
        assert out[i] in topk[i]
    # top-p → 0 degenerates to argmax
    out = hip().softmax_sample(logits, ones, offk, torch.full_like(ones, 1e-6), gen)
    assert torch.equal(out, logits.argmax(-1))
    # grammar mask respected
    mask = torch.zeros(B, V, dtype=torch.bool, device="cuda")
    mask[:, 7] = True
    mask[:, 100] = True
    out = hip().softmax_sample(logits, ones, offk, ones, gen, mask)
    assert all(int(t) in (7, 100) for t in out.tolist())


@requires_gpu
def test_model_forward_gpu_vs_cpu_reference():
    """Whole tiny model: GPU kernels vs CPU fp32 reference on identical
    weights — the kernels compose correctly."""
    from agentcontrolplane_amd.engine.batch import FlatBatch, SeqMeta
    from agentcontrolplane_amd.engine.config import PRESETS, EngineConfig
    from agentcontrolplane_amd.models.llama import LlamaForCausalLM

    ecfg = EngineConfig(model="tiny-gpu", num_kv_blocks=64, kv_block_size=16)
    mcfg = PRESETS["tiny-gpu"]
    gpu_model = LlamaForCausalLM(mcfg, ecfg, "cuda")
    gpu_model.random_init(0)
    gpu_model.allocate_kv_cache(64, 16)

    import dataclasses

    cpu_cfg = dataclasses.replace(mcfg, dtype="float32")
    cpu_model = LlamaForCausalLM(cpu_cfg, ecfg, "cpu")
    cpu_model.random_init(0)
    cpu_model.allocate_kv_cache(64, 16)
    # copy weights (fp32 promotion)
    cpu_model.embed = gpu_model.embed.cpu().float()
    cpu_model.lm_head = gpu_model.lm_head.cpu().float()
    cpu_model.final_norm = gpu_model.final_norm.cpu().float()
    for cl, gl in zip(cpu_model.layers, gpu_model.layers):
        for f in ("input_norm", "qkv", "o", "post_norm", "gate_up", "down"):
            setattr(cl, f, getattr(gl, f).cpu().float())

    T = 33
    tokens = torch.randint(0, mcfg.vocab_size, (T,))
    meta = SeqMeta(
        seq_id=1, query_len=T, seq_len=T, ctx_len=0,
        block_table=list(range(4)), needs_logits=True,
    )

    def make_batch(device):
        return FlatBatch(
            token_ids=tokens.to(device), positions=torch.arange(T, device=device),
            slot_mapping=torch.arange(T, device=device), prefills=[meta],
            num_prefill_tokens=T, decode_seq_ids=[], decode_block_tables=None,
            decode_seq_lens=None,
            logit_rows=torch.tensor([T - 1], device=device), sample_seq_ids=[1],
        )

    glog = gpu_model.forward(make_batch("cuda")).cpu()
    clog = cpu_model.forward(make_batch("cpu"))
    scale = clog.abs().max().item()
    err = (glog - clog).abs().max().item()
    assert err / max(scale, 1e-6) < 0.08, f"rel err {err / scale} (scale {scale})"


@requires_gpu
@pytest.mark.parametrize(
    "m,n,k",
    [
        (256, 256, 128),      # a single tile, two chunks
        (300, 512, 256),      # ragged M (row-clamp + store guard)
        (1024, 1536, 4096),   # multi-tile, deep K
        (2048, 768, 1664),    # K % 128 == 0 but K % 256 != 0; odd tile grid
    ],
)
def test_gemm_bf16(m, n, k):
    """The own products by threshold, on the largest tiles, vs fp32 matmul oracle."""
    torch.manual_seed(11)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(n, k, device="cuda", dtype=torch.bfloat16)
    got = hip().gemm_bf16(x, w)
    want = x.float() @ w.float().t()
    # bf16 inputs, fp32 accumulation: error scales with sqrt(K)
    tol = 0.03 * math.sqrt(k)  # bf16 output rounding of ~4.5σ results
    assert maxerr(got, want) < tol, maxerr(got, want)


@requires_gpu
@pytest.mark.parametrize("block", [16, 64])
@pytest.mark.parametrize("B,lo,hi,shared,kv", [
    (2, 900, 1000, 640, 8), (3, 2000, 4000, 1920, 2), (70, 300, 900, 320, 8), (200, 700, 1100, 640, 8),
    (40, 300, 1100, 64, 32),
])
def test_decode_over_shared_pages(B, lo, hi, shared, kv, block):
    """Sequences that begin alike read the same pages, by other loads: as from pages of their own.
    Two beginnings take turns, one sequence has neither."""
    gen = torch.Generator("cuda").manual_seed(B)
    lens = torch.randint(lo, hi + 1, (B,), generator=gen, device="cuda", dtype=torch.int32)
    pages, head = -(-hi // block), shared // block
    own = torch.randperm(B * pages, generator=gen, device="cuda").int().view(B, pages)
    caches = [torch.randn(B * pages, block, kv, 128, generator=gen, device="cuda").bfloat16()
              for _ in range(2)]
    tables = own.clone()
    for s in range(2, B - 1):
        tables[s, :head] = own[s % 2, :head]
        for cache in caches:
            cache[own[s, :head].long()] = cache[own[s % 2, :head].long()]
    H = min(32, 8 * kv)
    q = torch.randn(B, H, 128, generator=gen, device="cuda").bfloat16()
    run = hip().attention_decode_raw
    got, want = (run(q, *caches, t, lens, 128 ** -0.5) for t in (tables, own))
    assert torch.equal(got, want)
    s = B // 2
    k, v = (c[own[s].long()].flatten(0, 1)[: lens[s]].double() for c in caches)
    k, v = (t.repeat_interleave(H // kv, 1) for t in (k, v))
    w = torch.softmax(torch.einsum("hd,khd->hk", q[s].double(), k) * 128 ** -0.5, -1)
    assert maxerr(got[s], torch.einsum("hk,khd->hd", w, v)) < 0.01


@requires_gpu
@pytest.mark.parametrize("m,n,k,at", [
    (75000, 256, 14336, (0, 74751, 74752, 74999)), (3, 152064, 8192, (0, 130815, 130816, 152063)),
    (0, 256, 128, ()), (5, 256, 128, (0, 4)),
])
def test_linear_of_large_operands(m, n, k, at, monkeypatch):
    """The threshold for the own kernel's rows takes operands of 2 GiB and more, in blocks, and
    rows of no 16-byte units: rows and outputs at the blocks' edges against double precision."""
    monkeypatch.setattr(ops, "_GEMM_MIN_M", 0)
    gen = torch.Generator("cuda").manual_seed(k)
    x = torch.empty(m * k + 4, device="cuda", dtype=torch.bfloat16).normal_(generator=gen)
    w = torch.empty(n, k, device="cuda", dtype=torch.bfloat16).normal_(generator=gen)
    x = x[4:].view(m, k) if m == 5 else x[:-4].view(m, k)
    got = ops.linear(x, w)
    assert got.shape == (m, n)
    rows, outs = (slice(None), list(at)) if n > 256 else (list(at), slice(None))
    a, b = x[rows].double(), w[outs].double()
    exact, slack = a @ b.T, k * 2.0 ** -24 * (a.abs() @ b.abs().T)
    assert ((got[rows][:, outs].double() - exact).abs() <= 2.0 ** -8 * exact.abs() + slack).all()


@requires_gpu
@pytest.mark.parametrize("chunks", [16, 32])
def test_sample_fullvocab_chunks_keep_the_tail_in_64_bits(chunks):
    """A nucleus that reaches just past the largest logit, by what chunks' tails lose in 32 bits.
    Tail weights are 2^-18 and, too few of them in a chunk to round up, 2^-36, so that sums of a
    thread's tokens are exact."""
    V, each, few = 128256, 128256 // chunks, 960 // chunks
    log2e = torch.tensor(1.44269504, dtype=torch.float32)
    near = torch.arange(-40, 41, dtype=torch.float32)

    def logit_of(power):  # exp of it is 2^power
        x = power / log2e * (1 + near * 2.0 ** -24)
        return x[x * log2e == power][0].item()

    x = torch.full((V,), logit_of(-18.0))
    for c in range(chunks):
        x[c * each + 5 : c * each + 5 + few] = logit_of(-36.0)
    tail = (V - chunks * few - 2) * 2.0 ** -18 + chunks * few * 2.0 ** -36
    p = torch.tensor(1 / (1 + tail + 1e-3), dtype=torch.float32)
    x[0] = 0.0
    x[1] = math.log(1 / p.item() + 0.7e-8 - 1 - tail)
    one = torch.ones(1, device="cuda")
    out = torch.zeros(1, dtype=torch.long, device="cuda")
    hip()._C.sample_fullvocab(out, x.cuda().view(1, V), one, out.clone(), one * p.cuda(), one * 0.9999,
                              None, None, chunks)
    assert out.item() == 1


def test_sample_fullvocab_takes_chunks_where_plain_rows_gain():
    """Rows without a threshold were 5 to 28% faster in chunks at the first three sizes, and 3 to 80%
    slower at the last five, as are all others there."""
    from agentcontrolplane_amd import _C

    chunks = _C.sample_fullvocab_chunks
    assert chunks(1, 128256) == 32 and chunks(16, 100000) == 32 and chunks(64, 152064) == 16
    for rows, vocab in [(65, 128256), (190, 128256), (512, 152064), (8, 65536), (16, 32000)]:
        assert chunks(rows, vocab) == 0


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [513, 4099, 16384, 32000, 50257, 128256, 152064])
def test_sample_fullvocab_chunks(V, dtype):
    """Rows in chunks draw what a workgroup a row does: every kind of row, with masks, few distinct
    logits (more keys in a bucket than a list takes), thresholds beyond the head, infinities and
    NaN, greedy ties, a mask that leaves one token."""
    C = hip()._C
    gen = torch.Generator(device="cuda").manual_seed(V)
    B = 48
    x = torch.randn(B, V, generator=gen, device="cuda") * 2.5
    x[8:16] = (x[8:16]).round()
    x[16:20, ::3] = float("-inf")
    x[20, 5] = float("inf")
    x[21, V - 1] = float("nan")
    x[22:24] = 1.0
    x[24:28] *= 40
    i = torch.arange(B, device="cuda")
    temps = torch.where(i % 8 == 7, 0.0, 0.8)
    ks = torch.where((i % 4 == 1) | (i % 4 == 3), 50, 0)
    ks[40:44] = torch.tensor([1, V - 1, V, V // 2], device="cuda")
    ps = torch.where(i % 4 >= 2, 0.9, 1.0)
    ps[44:48] = torch.tensor([0.0, 1e-6, 0.99999, 0.5], device="cuda")
    u = torch.rand(B, generator=gen, device="cuda")
    mask = torch.rand(3, V, generator=gen, device="cuda") < 0.5
    mask[2] = False
    mask[2, V - 2] = True
    which = torch.where(i % 5 == 0, (i // 5) % 3, -1).int()
    x = x.to(dtype)
    for m, to in ((None, None), (mask, which)):
        outs = []
        for chunks in (0, 16, 32):
            out = torch.full((B,), -1, device="cuda")
            C.sample_fullvocab(out, x, temps, ks, ps, u, m, to, chunks)
            outs.append(out.tolist())
        assert outs[0] == outs[1] == outs[2]
        assert all(0 <= t < V for t in outs[0])
        if m is not None:
            assert all(mask[w, t] for w, t in zip(which.tolist(), outs[0]) if w >= 0)



@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("chunks", [0, 32])
def test_sample_fullvocab_mass_of_small_weights(dtype, chunks):
    """All weights are powers of two: 16384 of 1, next to each three of 2^-26, then groups of 1/2 and
    1/4, the last of which a top-p just reaches.  Their sum is exact in 64 bits, and the small ones,
    which are 7e-4 together, count: by fours in fp32 they are lost beside the 1, and so is the group."""
    C, n, V = hip()._C, 16384, 1 << 17
    T = torch.tensor(1.44269504)  # logits are octaves: 1 / T times log2 e rounds to 1
    assert T.reciprocal() * 1.44269504 == 1
    rows, ps, firsts = [], [], []
    for half in range(200, 1000, 40):
        for quarter in range(1000, 3000, 100):
            above = n + half / 2
            total = above + quarter / 4 + 3 * n * 2.0**-26
            p = torch.tensor(above / total)
            while float(p) * total <= above:
                p = torch.nextafter(p, torch.tensor(1.0))
            if 2e-5 < float(p) * total - above < 4e-4:
                rows.append([(half, -1.0), (quarter, -2.0)])
                ps.append(p)
                firsts.append((4 * n + half, above, above + quarter / 4))
    assert len(rows) >= 20
    x = torch.full((len(rows), V), float("-inf"))
    x[:, : 4 * n] = -26.0
    x[:, : 4 * n : 4] = 0.0
    for row, groups in zip(x, rows):
        at = 4 * n
        for count, value in groups:
            row[at : at + count] = value
            at += count
    out, u = torch.full((len(rows),), -1, device="cuda"), torch.full((len(rows),), 0.9995)
    C.sample_fullvocab(out, x.to("cuda", dtype), T.expand(len(rows)).contiguous().cuda(),
                       torch.zeros(len(rows), dtype=torch.long, device="cuda"),
                       torch.stack(ps).cuda(), u.cuda(), None, None, chunks)
    want = [at + int((float(u[0]) * total - above) * 4) for at, above, total in firsts]
    assert out.tolist() == want


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [8200, 32000, 128256, 262144])
@pytest.mark.parametrize("std", [0.05, 2.5, 8.0])
def test_sample_fullvocab_rows_by_units(V, std, dtype):
    """A row by units of 16 bytes, from a few of them a wave to more than its registers hold, against 64
    bits: logits over a part of an octave and over more than the buckets have, a few far above the rest,
    ones without weight, temperatures that take the boundary to either end.  Weights are rounded to 32
    bits, so one draw of 32 may fall between the two sums."""
    C, B = hip()._C, 32
    gen = torch.Generator(device="cuda").manual_seed(V)
    x = torch.randn(B, V, generator=gen, device="cuda") * std
    x[:4] *= 3
    x[4:6, :100] += 12
    x[6:8, ::7] = float("-inf")
    x[8] = x[8].abs()
    x = x.to(dtype)
    u, one = torch.rand(B, generator=gen, device="cuda"), torch.ones(B, device="cuda")
    mask = torch.rand(2, V, generator=gen, device="cuda") < 0.7
    which = (torch.arange(B, device="cuda") % 3 - 1).int()
    for t, k, p in [(0.8, 0, 1.0), (0.8, 1, 1.0), (0.8, 50, 1.0), (0.8, 7000, 1.0), (0.05, 40, 1.0),
                    (0.8, 0, 0.1), (0.8, 0, 0.95), (0.8, 0, 0.99), (0.8, 0, 0.999), (6.4, 0, 0.9),
                    (0.1, 0, 0.9), (0.8, 50, 0.95), (1.5, 3000, 0.6)]:
        for m, to in ((None, None), (mask, which)):
            out = torch.full((B,), -1, device="cuda")
            C.sample_fullvocab(out, x, one * t, (one * k).long(), one * p, u, m, to, 0)
            v = x.double()
            if m is not None:
                v = torch.where((which >= 0).view(-1, 1) & ~mask[which.clamp(min=0)], -torch.inf, v)
            keep = v >= v.topk(k, 1).values[:, -1:] if k else torch.ones_like(v, dtype=torch.bool)
            w = torch.where(keep, ((v - v.max(1, keepdim=True).values) / t).exp(), 0.0)
            if p < 1:
                top, order = w.sort(1, descending=True)
                ahead = top.cumsum(1) - top
                n = (ahead < (one * p).double().view(-1, 1) * w.sum(1, keepdim=True)).sum(1)
                least = v.gather(1, order).gather(1, n.view(-1, 1) - 1)
                w = torch.where(v >= least, w, 0.0)
            cdf = w.cumsum(1)
            if not k and p == 1:
                # the general path, whose sums are of 32 bits: V / 256 weights and then 256 stripes in
                # order, each rounded to 2^-24 of them, and the weights to less than 2^-18
                off = (V / 256 + 256) * 2.0**-24 + 2.0**-18
                to_here = (cdf / cdf[:, -1:]).gather(1, out.view(-1, 1)).view(-1)
                share = (w / cdf[:, -1:]).gather(1, out.view(-1, 1)).view(-1)
                assert bool(((to_here >= u - off) & (to_here - share <= u + off) & (share > 0)).all())
                continue
            want = (cdf > u.double().view(-1, 1) * cdf[:, -1:]).int().argmax(1)
            assert int((out != want).sum()) <= 1, (t, k, p, m is not None)
    out = torch.full((B,), -1, device="cuda")
    C.sample_fullvocab(out, x, one * 0, (one * 0).long(), one, u, None, None, 0)
    first = torch.where(x == x.max(1, keepdim=True).values, torch.arange(V, device="cuda"), V).min(1)
    assert torch.equal(out, first.values)


@requires_gpu
@pytest.mark.parametrize("V,chunks", [(600, 0), (32000, 0), (32001, 0), (128256, 0), (128256, 16)])
@pytest.mark.parametrize("masked", [False, True])
def test_sample_fullvocab_greedy_of_lowest_logits(V, chunks, masked):
    """The first of the largest logits, however low: -3.4e38, with which masks are written, is one."""
    C, B = hip()._C, 4
    x = torch.full((B, V), float("-inf"), device="cuda")
    first = [0, 77, V // 2, V - 1]
    for i, at in enumerate(first):
        x[i, at:] = -3.4e38
    x[1, 78:] = torch.finfo(torch.float32).min
    mask = torch.ones(B, V, dtype=torch.bool, device="cuda") if masked else None
    if masked:
        for i, at in enumerate(first):
            x[i, :at] = 1.0
            mask[i, :at] = False
    to = torch.arange(B, device="cuda").int() if masked else None
    out, zero = torch.full((B,), -1, device="cuda"), torch.zeros(B, device="cuda")
    C.sample_fullvocab(out, x, zero, zero.long(), zero + 1, zero, mask, to, chunks)
    assert out.tolist() == first


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [8200, 128256])
@pytest.mark.parametrize("std", [0.0, 0.02, 2.5])
def test_sample_fullvocab_few_allowed(V, std, dtype):
    """Masks that leave fewer tokens than a top-k, as many, and more, some of them of no weight, in a
    narrow range and all alike: against 64 bits, where one draw of a row's five may fall between sums."""
    C, gen = hip()._C, torch.Generator(device="cuda").manual_seed(V)
    counts = [1, 2, 49, 50, 51, 320, 321, 3000, 4097, 6000]
    B = len(counts)
    x = (torch.randn(B, V, generator=gen, device="cuda") * std + 0.0).to(dtype)  # and no -0
    mask = torch.zeros(B, V, dtype=torch.bool, device="cuda")
    for i, n in enumerate(counts):
        at = torch.randperm(V, generator=gen, device="cuda")[:n]
        mask[i, at] = True
        x[i, at[: n // 8]] = float("-inf")
    v = torch.where(mask, x.double(), -torch.inf)
    to, one = torch.arange(B, device="cuda").int(), torch.ones(B, device="cuda")
    finite = torch.where(v > -torch.inf, v, 0.0)
    for k in (1, 50, 4096, 4097, V - 1):
        keep = (v >= v.topk(k, 1).values[:, -1:]) & (v > -torch.inf)
        for p in (1.0, 0.9):
            w = torch.where(keep, ((finite - v.max(1, keepdim=True).values) / 0.8).exp(), 0.0)
            if p < 1:
                top, order = w.sort(1, descending=True)
                ahead = top.cumsum(1) - top
                n = (ahead < (one * p).double().view(-1, 1) * w.sum(1, keepdim=True)).sum(1)
                w = torch.where(v >= v.gather(1, order).gather(1, n.view(-1, 1) - 1), w, 0.0)
            cdf, off = w.cumsum(1), 0
            for _ in range(5):
                u = torch.rand(B, generator=gen, device="cuda")
                out = torch.full((B,), -1, device="cuda")
                C.sample_fullvocab(out, x, one * 0.8, (one * k).long(), one * p, u, mask, to, 0)
                assert bool(mask.gather(1, out.view(-1, 1)).all())
                want = (cdf > u.double().view(-1, 1) * cdf[:, -1:]).int().argmax(1)
                off += int((out != want).sum())
            assert off <= 1, (k, p)


@pytest.mark.gpu
def test_sample_fullvocab_vs_oracle():
    """csrc/sampling_fullvocab.hip vs the fp32 reference over a Llama-3
    sized vocabulary: greedy exact, draws match the oracle's inverse CDF
    for given uniforms, top-k/top-p respect the oracle's kept sets, and
    compact masks (mask_map indirection) are honored exactly."""
    from agentcontrolplane_amd.ops import reference

    torch.manual_seed(0)
    device = "cuda"
    B, V = 64, 128256
    gen = torch.Generator(device=device)
    logits = torch.randn(B, V, device=device, dtype=torch.float32) * 3
    uniforms = torch.rand(B, device=device)
    zeros = torch.zeros(B, device=device)
    ones = torch.ones(B, device=device)
    offk = torch.zeros(B, dtype=torch.long, device=device)

    # greedy: exact argmax match
    out = hip().softmax_sample(logits, zeros, offk, ones, gen, uniforms=uniforms)
    assert torch.equal(out, logits.argmax(-1))

    # temperature-only fp32: draws match the oracle inverse CDF
    ref = reference.softmax_sample(
        logits.cpu(), ones.cpu() * 0.8, offk.cpu(), ones.cpu(), None,
        uniforms=uniforms.cpu())
    out = hip().softmax_sample(logits, ones * 0.8, offk, ones, gen,
                               uniforms=uniforms)
    frac = (out.cpu() == ref).float().mean().item()
    assert frac >= 0.95, f"only {frac:.2%} of draws matched the oracle"

    # top-k: every draw inside the oracle's kept set {x >= kth}
    k = 50
    out = hip().softmax_sample(logits, ones, torch.full_like(offk, k), ones,
                               gen, uniforms=uniforms)
    kth = torch.topk(logits, k, dim=-1).values[:, -1]
    picked = logits[torch.arange(B, device=device), out]
    assert (picked >= kth - 1e-6).all()

    # top-p: draws inside the oracle nucleus
    p = 0.7
    out = hip().softmax_sample(logits, ones, offk, ones * p, gen,
                               uniforms=uniforms)
    probs = torch.softmax(logits, -1)
    sp, si = torch.sort(probs, descending=True, dim=-1)
    cum = sp.cumsum(-1)
    for i in range(B):
        keep_n = int((cum[i] - sp[i] <= p).sum())
        kept = set(si[i, :max(1, keep_n)].tolist())
        assert int(out[i]) in kept

    # bf16 logits path + compact mask rows with indirection
    lb = logits.bfloat16()
    n_masked = 8
    mask = torch.zeros(n_masked, V, dtype=torch.bool, device=device)
    allowed_ids = torch.randint(0, V, (n_masked, 37), device=device)
    for j in range(n_masked):
        mask[j, allowed_ids[j]] = True
    mask_map = torch.full((B,), -1, dtype=torch.int32, device=device)
    mask_map[: n_masked] = torch.arange(n_masked, dtype=torch.int32, device=device)
    out = hip().softmax_sample(lb, ones, offk, ones, gen, mask,
                               uniforms=uniforms, mask_map=mask_map)
    for j in range(n_masked):
        assert bool(mask[j, out[j]]), "masked row sampled a disallowed token"
    # unmasked rows unaffected by the compact mask
    out_ref = hip().softmax_sample(lb, ones, offk, ones, gen,
                                   uniforms=uniforms)
    assert torch.equal(out[n_masked:], out_ref[n_masked:])


@pytest.mark.gpu
def test_tp_shard_path_math_on_gpu():
    """TP assembly path on one GPU (driver-checkable without multi-GPU):
    a world=1 'shard' built through shard_from_full + the all_reduce hook
    must equal the plain model exactly, and world=2 shards must run the
    CDNA4 kernels at halved head counts without shape faults (the gloo
    CPU test proves the world=2 math)."""
    import dataclasses

    from agentcontrolplane_amd.engine.batch import FlatBatch, SeqMeta
    from agentcontrolplane_amd.engine.config import PRESETS, EngineConfig
    from agentcontrolplane_amd.models.llama import LlamaForCausalLM
    from agentcontrolplane_amd.parallel.tp import shard_from_full

    cfg = dataclasses.replace(PRESETS["tiny-gpu"])
    ecfg = EngineConfig(model="tiny-gpu", device="cuda", num_kv_blocks=64)
    torch.manual_seed(0)
    full = LlamaForCausalLM(cfg, ecfg, "cuda")
    full.random_init(0)
    full.allocate_kv_cache(64, 16)

    T = 24
    g = torch.Generator().manual_seed(42)
    tokens = torch.randint(0, cfg.vocab_size, (T,), generator=g).cuda()
    meta = SeqMeta(seq_id=1, query_len=T, seq_len=T, ctx_len=0,
                   block_table=[0, 1], needs_logits=True)

    def mk():
        return FlatBatch(
            token_ids=tokens.clone(), positions=torch.arange(T, device="cuda"),
            slot_mapping=torch.arange(T, device="cuda"), prefills=[meta],
            num_prefill_tokens=T, decode_seq_ids=[],
            decode_block_tables=None, decode_seq_lens=None,
            logit_rows=torch.tensor([T - 1], device="cuda"), sample_seq_ids=[1],
        )

    ref_logits = full.forward(mk()).float()

    shard1 = LlamaForCausalLM(cfg, ecfg, "cuda", tp_rank=0, tp_world=1)
    shard_from_full(full, shard1, 0, 1)
    shard1.allocate_kv_cache(64, 16)
    shard1.all_reduce = lambda t: t  # world=1 collective = identity
    out1 = shard1.forward(mk()).float()
    assert torch.equal(out1, ref_logits), "world=1 shard path diverged"

    # world=2 shards: halved Hq/Hkv shapes through the HIP kernels
    for rank in (0, 1):
        sh = LlamaForCausalLM(cfg, ecfg, "cuda", tp_rank=rank, tp_world=2)
        shard_from_full(full, sh, rank, 2)
        sh.allocate_kv_cache(64, 16)
        sh.all_reduce = lambda t: t  # partial sums: shape/sanity only
        out = sh.forward(mk()).float()
        assert out.shape == ref_logits.shape
        assert torch.isfinite(out).all()


@pytest.mark.gpu
def test_attention_bias_serving_on_gpu():
    """Qwen2-style QKV bias through the CDNA4 kernel path: the bias add
    precedes the strided q/k/v views, so the fused-QKV stride handling
    must hold on the result tensor."""
    from agentcontrolplane_amd.engine.config import EngineConfig
    from agentcontrolplane_amd.engine.engine import InferenceEngine
    from agentcontrolplane_amd.engine.request import SamplingParams

    eng = InferenceEngine(
        EngineConfig(model="tiny-gpu-bias", device="cuda", num_kv_blocks=128),
        start=True,
    )
    try:
        assert eng.model.layers[0].qkv_bias is not None
        res = eng.chat(
            [{"role": "user", "content": "bias check"}],
            sampling=SamplingParams(max_tokens=8, temperature=0.8),
        )
        assert res.completion_tokens <= 8
    finally:
        eng.stop()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 2, 4])
@pytest.mark.parametrize("n,k,kind", [
    (1, 32, "plain"), (17, 96, "bias"), (16, 288, "strided"), (250, 1120, "bias"),
    (4096, 4096, "plain"), (33, 8160, "strided"), (16, 64, "glu"), (80, 2976, "glu"),
    (1504, 4096, "glu"),
])
def test_step_linear(m, n, k, kind):
    """A few rows' products, against double precision: one rounding of the sum to 16 bits, and
    sums of k terms in 32 bits."""
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=gen).bfloat16().cuda()
    w = torch.randn(n, k + 16, generator=gen).bfloat16().cuda()
    x, w = (x[:, 8:], w[:, :k]) if kind == "strided" else (x[:, :k].clone(), w[:, :k].clone())
    bias = torch.randn(n, generator=gen).bfloat16().cuda() if kind == "bias" else None
    assert ops._few_rows(x, w, bias)
    exact = x.double() @ w.double().T + (0 if bias is None else bias.double())
    # sums: k terms of at most |x||w|, 2^-24 each
    slack = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    if kind != "glu":
        got = ops.step_linear(x, w, bias).double()
        assert ((got - exact).abs() <= 2.0 ** -8 * exact.abs() + slack + 1e-30).all()
        return
    got = ops.step_linear_swiglu(x, w).double()
    g, u = exact.chunk(2, 1)
    # both halves are off by a rounding and the sums' slack; silu's slope is at most 1.1
    dg, du = (2.0 ** -8 * t.abs() + s for t, s in zip((g, u), slack.chunk(2, 1)))
    silu = torch.nn.functional.silu(g)
    bound = 1.1 * dg * (u.abs() + du) + silu.abs() * du
    want = silu * u
    assert ((got - want).abs() <= bound + 2.0 ** -7 * want.abs() + 1e-30).all()


@pytest.mark.gpu
def test_step_linear_leaves_other_forms():
    """What its kernel does not take goes the way of linear(), with the same result or error."""
    x = torch.randn(4, 4104, device="cuda").bfloat16()
    w = torch.randn(64, 4096, device="cuda").bfloat16()
    lin = torch.nn.functional.linear
    for a, b in [
        (torch.randn(5, 4096, device="cuda").bfloat16(), w),
        (x[:, 1:4097], w), (x[:, :4104:2][:, :2048], w[:, :2048]),
        (x[:, :4096].float(), w.float()), (x[:0, :4096], w),
        (x[:, :40], w[:, :40]), (x[:, :4096], w.T.contiguous().T), (x[:, None, :4096], w),
    ]:
        assert not ops._few_rows(a, b)
        assert torch.equal(ops.step_linear(a, b), lin(a, b))
    with pytest.raises(RuntimeError):
        ops.step_linear(x[:, :4096], w[:, :2048])


@pytest.mark.gpu
@pytest.mark.parametrize("needs", ["x", "w", "bias"])
def test_step_linear_keeps_gradients(needs):
    """A few rows that autograd records get the derivatives that linear() gives."""
    gen = torch.Generator().manual_seed(3)
    shape = {"x": (4, 256), "w": (64, 256), "bias": (64,)}
    t = {n: torch.randn(*s, generator=gen).bfloat16().cuda() for n, s in shape.items()}
    t[needs].requires_grad_()
    got, = torch.autograd.grad(ops.step_linear(t["x"], t["w"], t["bias"]).float().sum(), t[needs])
    want, = torch.autograd.grad(
        torch.nn.functional.linear(t["x"], t["w"], t["bias"]).float().sum(), t[needs]
    )
    assert torch.equal(got, want)
    with torch.no_grad():
        assert ops._few_rows(t["x"], t["w"], t["bias"])
