"""Products of many rows (csrc/linear.hip): every tile at its edges against double precision,
and which calls its rule takes."""
import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode

from agentcontrolplane_amd import ops
from agentcontrolplane_amd.engine.config import ClampedGluSpec

TILES = range(14)


def operands(m, n, k, seed, strided=False):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k + 8, generator=gen).bfloat16().cuda()
    w = torch.randn(n, k + 16, generator=gen).bfloat16().cuda()
    if strided:
        return x[:, 8:], w[:, :k]
    return x[:, :k].clone(), w[:, :k].clone()


def sums(x, w, bias=None):
    """The product in 64 bits, and what sums of k terms in 32 bits may be off."""
    exact = x.double() @ w.double().T + (0 if bias is None else bias.double())
    return exact, x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k,splits,kind", [
    (1, 8, 64, 1, "plain"), (33, 264, 128, 2, "bias"), (255, 520, 192, 3, "strided"),
    (257, 248, 64, 1, "bias"), (600, 1304, 320, 1, "strided"), (5, 1032, 4096, 64, "plain"),
    (2300, 3080, 128, 1, "bias"),
])
def test_linear(tile, m, n, k, splits, kind):
    """One rounding of the sum to 16 bits, and sums of k terms in 32 bits; nothing is written
    beside the outputs.  The last case has several of the smaller tiles a workgroup."""
    hip = ops._hip()
    x, w = operands(m, n, k, m + n + k, kind == "strided")
    bias = torch.randn(n, device="cuda").bfloat16() if kind == "bias" else None
    pad = torch.full((m + 2, n + 16), 7.0, device="cuda").bfloat16()
    out = pad[1:-1, 8:-8]
    hip.linear(x, w, bias, out=out, tile=tile, splits=splits)
    exact, slack = sums(x, w, bias)
    assert ((out.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + slack + 1e-30).all()
    pad[1:-1, 8:-8] = 7.0
    assert (pad == 7.0).all()


FORMS = {"swiglu": (0.0,) * 4, "glu": (7.0, 1.702, 1.0, 0.0)}  # limit, alpha, offset, cubic


def check_gated(got, x, w, unit):
    exact, slack = sums(x, w)
    g, u = exact.chunk(2, 1)
    # both halves are off by a rounding and the sums' slack
    dg, du = (2.0 ** -8 * t.abs() + s for t, s in zip((g, u), slack.chunk(2, 1)))
    alpha, plus = (1.702, 1.0) if unit == "glu" else (1.0, 0.0)
    if unit == "glu":
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
    act = g * torch.sigmoid(alpha * g)  # slope at most 1.1 for any alpha
    want = act * (u + plus)
    bound = 1.1 * dg * (u.abs() + du + plus) + act.abs() * du
    assert ((got.double() - want).abs() <= bound + 2.0 ** -7 * want.abs() + 1e-30).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k,splits,unit", [
    (1, 16, 64, 1, "swiglu"), (65, 272, 128, 2, "glu"), (260, 784, 192, 1, "glu"),
    (513, 1552, 320, 1, "swiglu"), (33, 2064, 256, 4, "swiglu"),
])
def test_linear_gated(tile, m, n, k, splits, unit):
    hip = ops._hip()
    if splits == 1 and not hip._C.linear_fits(tile, True):
        with pytest.raises(RuntimeError):
            hip.linear(*operands(m, n, k, 1), unit=unit, tile=tile)
        return
    x, w = operands(m, n, k, m + n + k)
    check_gated(hip.linear(x, w, None, unit, FORMS[unit], tile=tile, splits=splits), x, w, unit)


#: outputs and rows of the tiles
SIZES = [(256, 256), (256, 224), (256, 192), (256, 160), (256, 128), (128, 192), (128, 128),
         (128, 96), (128, 64), (128, 32), (192, 128), (64, 64), (64, 32), (128, 160)]


@pytest.mark.parametrize("m,n,k,glu,parts,want", [
    (2500, 28672, 4096, True, False, ((256, 160), 1)),
    (6000, 28672, 4096, True, False, ((256, 224), 1)),
    (7664, 16384, 2048, True, False, ((256, 192), 1)),
    (10000, 6144, 4096, False, False, ((256, 192), 1)),
    (10000, 12288, 4096, False, True, ((256, 192), 1)),
    (160, 28672, 4096, True, False, ((128, 160), 1)),
    (190, 4096, 14336, False, True, ((128, 192), 8)),
    # tiles that are whole in the inner dimension, or large ones in parts, were 15 to 26% slower
    (190, 5120, 5120, False, True, ((128, 96), 3)),
    (777, 4096, 4096, False, False, ((128, 128), 1)),
    (128, 5120, 5120, False, False, ((128, 64), 3)),
    (256, 3072, 3072, False, True, ((128, 96), 3)),
])
def test_choice_of_tiles(m, n, k, glu, parts, want):
    """Measured to be the faster one of two models' choices; above 2100 rows it is by the fragments
    alone, which the step times of few rows do not speak for."""
    tile, splits = ops._hip()._C.linear_choice(m, n, k, glu, parts)
    assert (SIZES[tile], splits) == want


@pytest.mark.parametrize("m", [1, 33, 2100, 2101, 2600, 2601, 1 << 20, (1 << 30) - 1])
@pytest.mark.parametrize("n,k", [(8, 64), (16, 320), (4104, 4096), (1 << 20, 64), (64, 1 << 20)])
@pytest.mark.parametrize("glu,parts", [(False, False), (True, False), (False, True)])
def test_choice_is_of_what_there_is(m, n, k, glu, parts):
    C = ops._hip()._C
    tile, splits = C.linear_choice(m, n, k, glu, parts)
    assert 0 <= tile < len(SIZES) and 1 <= splits <= k // 64
    assert C.linear_fits(tile, glu and splits == 1)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [None, (7.0, 1.702, 1.0, 0.0), (1e30, 1.0, 0.0, 0.0),
                                  (3e38, 1.5957691, 0.0, 0.044715)])
def test_gated_unit_of_every_gate(form):
    """All 65536 gates of 16 bits, zeros, denormals, infinities and what is no number among them, come out
    as from the unit's own pass, beside their like and beside ordinary ones."""
    hip, n = ops._hip(), 1 << 16
    gates = torch.arange(n, device="cuda").short().view(torch.bfloat16)
    for order in (gates, gates[torch.randperm(n, device="cuda")]):
        w = torch.zeros(2 * n, 64, device="cuda", dtype=torch.bfloat16)
        w[:n, 0], w[n:, 0] = order, torch.linspace(-3, 3, n, device="cuda").bfloat16()
        x = torch.zeros(33, 64, device="cuda", dtype=torch.bfloat16)
        x[:, 0] = 1.0
        y = hip.linear(x, w, tile=6)
        if form is None:
            got, want = hip.linear(x, w, unit="swiglu", tile=6), ops.swiglu(y)
        else:
            got = hip.linear(x, w, None, "glu", form, tile=6)
            want = torch.empty_like(got)
            ops.clamped_glu(y, *form[:3], want, form[3])
        nan = want.isnan()
        assert torch.equal(got.isnan(), nan) and torch.equal(got[~nan], want[~nan])


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("k", [64, 128, 192, 320])
def test_linear_of_several_tiles_a_workgroup(tile, k):
    """The large tiles, one workgroup a CU: the loads run ahead over the end of a tile of 1, 2, 3
    and 5 chunks, into ragged rows and outputs, behind every kind of store."""
    hip, m, n = ops._hip(), 4200, 8208
    assert -(-m // SIZES[tile][1]) * -(-n // SIZES[tile][0]) > 2 * 256
    x, w = operands(m, n, k, k)
    exact, slack = sums(x, w)
    got = hip.linear(x, w, tile=tile).double()
    assert ((got - exact).abs() <= 2.0 ** -8 * exact.abs() + slack + 1e-30).all()
    bias = torch.randn(n, device="cuda").bfloat16()
    exact += bias.double()
    got = hip.linear(x, w, bias, tile=tile).double()
    assert ((got - exact).abs() <= 2.0 ** -8 * exact.abs() + slack + 1e-30).all()
    for unit in FORMS:
        check_gated(hip.linear(x, w, None, unit, FORMS[unit], tile=tile), x, w, unit)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("n,k", [(8208, 4096), (65552, 512), (1040, 32320)])
def test_linear_of_large_weights_and_one_tile_of_rows(tile, n, k):
    """Those that no other workgroup reads pass by the caches, in kernels of their own, and tiles
    begin apart in the inner dimension: plain, bias, both units and parts, at the smallest weights
    that take them, several tiles a workgroup, fewer tiles than chunks."""
    hip, m = ops._hip(), SIZES[tile][1] - 6
    assert n * k >= 32 << 20 > (n - 32) * k
    x, w = operands(m, n, k, m)
    exact, slack = sums(x, w)
    bias = torch.randn(n, device="cuda").bfloat16()
    for splits in (1, 3):
        got = hip.linear(x, w, tile=tile, splits=splits).double()
        assert ((got - exact).abs() <= 2.0 ** -8 * exact.abs() + slack).all()
        got, want = hip.linear(x, w, bias, tile=tile, splits=splits).double(), exact + bias.double()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + slack).all()
        for unit in FORMS:
            if splits > 1 or hip._C.linear_fits(tile, True):
                check_gated(hip.linear(x, w, None, unit, FORMS[unit], tile=tile, splits=splits),
                            x, w, unit)
    parts = hip._C.linear_parts(x, w, tile, 3)
    assert parts.shape == (3, m, n) and ((parts.double().sum(0) - exact).abs() <= slack).all()


@pytest.mark.gpu
@pytest.mark.parametrize("unit", ["swiglu", "glu"])
@pytest.mark.parametrize("splits", [1, 2])
def test_gated_unit_is_that_of_two_passes(unit, splits):
    """Bit for bit: a unit with fewer bits than the passes apart have shows in some of a million
    outputs.  The products' sums do not depend on the tile."""
    hip = ops._hip()
    x, w = operands(600, 4096, 256, 5)
    form = (3.0, 1.702, 1.0, 0.0) if unit == "glu" else (0.0,) * 4
    for tile in TILES:
        if splits == 1 and not hip._C.linear_fits(tile, True):
            continue
        y = hip.linear(x, w, tile=tile, splits=splits)
        got = hip.linear(x, w, None, unit, form, tile=tile, splits=splits)
        want = torch.empty_like(got)
        if unit == "glu":
            ops.clamped_glu(y, *form[:3], want)
        else:
            want = ops.swiglu(y)
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(5, 4096, 512), (100, 2048, 1024), (700, 2056, 1024),
                                   (3000, 1024, 2048)])
def test_step_linear_takes_its_rows(m, n, k):
    """The public entry goes to the kernel, in a graph as well, whose replays see new inputs."""
    x, w = operands(m, n, k, m)
    assert ops._many_rows(x, w)
    got = ops.step_linear(x, w)
    assert torch.equal(got, ops._hip().linear(x, w))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.step_linear(x, w)
    for seed in range(3):
        x.copy_(operands(m, n, k, 100 + seed)[0])
        graph.replay()
        assert torch.equal(y, ops.step_linear(x, w))


@pytest.mark.gpu
def test_linear_from_several_threads():
    """Every thread may be the first to launch a kernel, each on a stream of its own."""
    from concurrent.futures import ThreadPoolExecutor

    x, w = operands(70, 264, 320, 9)
    torch.cuda.synchronize()

    def run(first):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            outs = [ops._hip().linear(x, w, tile=(first + i) % len(TILES)) for i in TILES]
        stream.synchronize()
        return outs

    with ThreadPoolExecutor(6) as pool:
        results = list(pool.map(run, range(6)))
    for outs in results:
        for out in outs:
            assert torch.equal(out, results[0][0])


@pytest.mark.gpu
def test_linear_leaves_other_forms():
    """What the kernel does not take, and what others follow, stays with the library."""
    x, w = operands(64, 2048, 1024, 0)
    lin = torch.nn.functional.linear
    assert ops._many_rows(x, w)
    base = torch.zeros(64 * 1032, device="cuda").bfloat16()
    for a, b in [
        (x.float(), w.float()), (x.half(), w.half()), (x[:, None], w), (x[:0], w),
        (x[:, :1000], w[:, :1000].contiguous()), (x, w[:2044]), (x.T.contiguous().T, w),
        (base[: 64 * 1026].view(64, 1026)[:, :1024], w), (base[1 : 1 + 65536].view(64, 1024), w),
        (x, w.T.contiguous().T),
    ]:
        assert not ops._many_rows(a, b)
        assert torch.equal(ops.step_linear(a, b), lin(a, b))
    assert ops._many_rows(x[:1].expand(64, 1024), w)  # a row stride of 0
    with pytest.raises(RuntimeError):
        ops.step_linear(x, w[:, :512])
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        tangent = torch.autograd.forward_ad.unpack_dual(ops.step_linear(dual, w)).tangent
    assert torch.equal(tangent, lin(torch.ones_like(x), w))
    each = torch.func.vmap(lambda t: ops.step_linear(t, w))(torch.stack([x, x + 1]))
    assert each.shape == (2, 64, 2048)
    w.requires_grad_()
    ops.step_linear(x, w).float().sum().backward()
    assert w.grad is not None


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 4096, 14336), (4, 6144, 4096), (2, 2048, 64), (64, 2048, 1024)])
def test_what_follows_the_library_sees_products(m, n, k):
    """Forward-mode derivatives, vmap, traces, dispatch modes and autocast, of few rows and many."""
    x, w = operands(m, n, k, m)
    lin = torch.nn.functional.linear
    assert ops._few_rows(x, w) if m <= 4 else ops._many_rows(x, w)
    ones = torch.ones_like(x)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, ones)
        tangent = torch.autograd.forward_ad.unpack_dual(ops.step_linear(dual, w)).tangent
        assert tangent is not None and torch.equal(tangent, lin(ones, w))
    assert torch.equal(torch.func.jvp(lambda t: ops.step_linear(t, w), (x,), (ones,))[1],
                       lin(ones, w))
    each = torch.func.vmap(lambda t: ops.step_linear(t, w))(torch.stack([x, x + 1]))
    assert each.shape == (2, m, n)
    traced = torch.jit.trace(lambda t: ops.step_linear(t, w), (x,), check_trace=False)
    assert torch.equal(traced(ones), lin(ones, w))
    with FlopCounterMode(display=False) as flops:
        ops.step_linear(x, w)
    assert flops.get_total_flops() == 2 * m * n * k
    with torch.autocast("cuda", torch.float16):
        y, want = ops.step_linear(x, w), lin(x, w)
    assert y.dtype == torch.float16 and torch.equal(y, want)


def test_rule_of_many_rows():
    """Few rows and small weights stay where they were; so does what the library is faster at."""
    pay = ops._many_rows_pay
    assert not pay(4, 4096, 4096, False) and pay(5, 4096, 4096, False)
    assert not pay(64, 2048, 64, False)
    assert not pay(8192, 4096, 4096, False) and pay(8192, 8192, 4096, True)
    assert pay(10000, 4096, 4096, False) and pay(16000, 4096, 14336, False)
    # where the library was as fast to 20% faster, but for a launch that parts take to be added up
    for m, n, k in [(8, 6144, 4096), (32, 7168, 4096), (16, 4096, 8192), (5, 8192, 8192),
                    (8, 2048, 8192), (61, 4096, 4096), (33, 3584, 3584),
                    (80, 2048, 4096), (96, 12288, 4096), (128, 13824, 5120), (1400, 32000, 4096)]:
        assert not pay(m, n, k, False) and pay(m, n, k, False, True) and pay(m, n, k, True)
    # where it was 3 to 150% slower
    for m, n, k in [(16, 4096, 4096), (32, 4096, 11008), (32, 2048, 8192), (13, 12288, 4096),
                    (40, 6144, 4096), (61, 4096, 14336), (5, 128256, 4096), (24, 128256, 4096),
                    (32, 256000, 2048), (61, 128256, 4096), (96, 4096, 8192),
                    (192, 12288, 4096), (96, 16448, 4096), (1739, 32000, 4096)]:
        assert pay(m, n, k, False)
    # not on the CPU
    x, w = torch.zeros(64, 1024).bfloat16(), torch.zeros(2048, 1024).bfloat16()
    assert not ops._many_rows(x, w)
    out = torch.empty(64, 1024).bfloat16()
    ops.step_linear_glu(x + 1, w + 0.01, ClampedGluSpec(1024, 7.0, 1.702, 1.0), out)
    want = torch.empty_like(out)
    ops.clamped_glu(ops.linear(x + 1, w + 0.01), 7.0, 1.702, 1.0, want)
    assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile,splits", [
    (1, 8, 128, 11, 2), (61, 4096, 4096, 6, 4), (190, 4096, 1024, 6, 3), (13, 9224, 448, 12, 5),
    (1100, 16384, 128, 0, 2), (3, 520, 192, 9, 3), (7, 16392, 256, 12, 4),
])
def test_parts_into_the_norm(m, n, k, tile, splits):
    """As the parts' own sum and the norm of it: the same roundings, in the same order."""
    hip = ops._hip()
    x, w = operands(m, n, k, m + n)
    gen = torch.Generator().manual_seed(n)
    residual = torch.randn(m, n, generator=gen).bfloat16().cuda()
    weight = torch.rand(n, generator=gen).bfloat16().cuda()
    parts = hip._C.linear_parts(x, w, tile, splits)
    if n > hip._C.ADD_RMSNORM_MOST:
        with pytest.raises(RuntimeError):
            hip._C.parts_add_rmsnorm(residual.clone(), residual, parts, weight, 1e-5)
        return
    y = parts if parts.dim() == 2 else hip.linear(x, w, tile=tile, splits=splits)
    sums = residual.clone()
    got = torch.empty_like(residual)
    if parts.dim() == 3:
        hip._C.parts_add_rmsnorm(got, sums, parts, weight, 1e-5)
    else:
        hip._C.fused_add_rmsnorm(got, sums, y, weight, 1e-5)
    new = (y.float() + residual.float()).bfloat16()
    assert torch.equal(sums, new)
    want = new.double() * torch.rsqrt((new.double() ** 2).mean(-1, keepdim=True) + 1e-5)
    # one rounding of the result, and sums of n squares in 32 bits
    assert ((got.double() - want * weight.double()).abs() <=
            (2.0 ** -8 + n * 2.0 ** -24) * (want * weight.double()).abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,heads,kv,d,k,tile,splits", [
    (1, 1, 1, 128, 128, 11, 2), (61, 32, 8, 128, 256, 5, 3), (13, 4, 4, 256, 448, 12, 5),
    (300, 2, 1, 512, 64, 0, 1),
])
def test_parts_into_the_caches(m, heads, kv, d, k, tile, splits):
    """Queries and cached rows are those of the sum's own pass and a rotation a head at a time."""
    hip = ops._hip()
    x, w = operands(m, (heads + 2 * kv) * d, k, m)
    gen = torch.Generator(device="cuda").manual_seed(d)
    angles = torch.rand(2 * 50 * (d // 2) + 1, generator=gen, device="cuda")
    aside = angles[1:].view(2, 50, d // 2)  # rows of no 16-byte units
    tables = aside.clone()
    pos = torch.randint(0, 50, (m,), generator=gen, device="cuda")
    slots = torch.randperm(m + 9, generator=gen, device="cuda")[:m]

    def caches():
        return [torch.zeros(m + 9, kv, d, dtype=torch.bfloat16, device="cuda") for _ in range(2)]

    y = hip.linear(x, w, tile=tile, splits=splits).view(m, heads + 2 * kv, d)
    results = []
    for cos_sin in (aside, tables):
        q, key, v = (t.clone() for t in y.split([heads, kv, kv], 1))
        results.append((q, *caches()))
        hip.rope_and_cache(q, key, v, pos, slots, *results[-1][1:], cos_sin)
    parts = hip._C.linear_parts(x, w, tile, splits)
    if parts.dim() == 3:
        results.append((torch.empty_like(results[0][0]), *caches()))
        to = results[-1]
        hip._C.rope_cache(to[0], None, None, pos, slots, *to[1:], tables, parts)
    for other in results[1:]:
        for a, b in zip(results[0], other):
            # the compiler may round a product before the sum in one of two kernels
            assert ((a.float() - b.float()).abs() <= 2.0 ** -7 * a.float().abs() + 1e-6).all()
        assert torch.equal(results[0][2], other[2])


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 61, 190, 2100])
def test_step_linear_with_what_follows(m):
    """The entries are the passes one after another, but for the product's sums of 32 bits, which
    may round to the next 16-bit value: an ulp, up to 2^-7 of it, and so may what follows."""
    x, w = operands(m, 2048, 1024, m)
    y, slack = sums(x, w)
    residual = x.repeat(1, 2)
    weight = torch.rand(2048, device="cuda").bfloat16()
    ulp = 2.0 ** -7
    dy = ulp * y.abs() + 2 * slack
    got, total = ops.step_linear_add_rmsnorm(x, w, residual.clone(), weight)
    want, new = ops.fused_add_rmsnorm(ops.step_linear(x, w), residual.clone(), weight)
    new = new.double()
    dt = dy + ulp * new.abs()
    assert ((total.double() - new).abs() <= dt).all()
    inv = torch.rsqrt((new ** 2).mean(-1, keepdim=True) + 1e-5)
    # the norm moves by its share of what its squares do
    turn = inv ** 2 * (2 * new.abs() * dt).mean(-1, keepdim=True) / 2
    bound = inv * weight.double() * (dt + new.abs() * turn) + ulp * want.double().abs()
    assert ((got.double() - want.double()).abs() <= bound).all()
    cos_sin = torch.rand(2, 9, 64, device="cuda")
    pos, slots = torch.arange(m, device="cuda") % 9, torch.arange(m, device="cuda")
    both = []
    for fused in (True, False):
        kc, vc = (torch.zeros(m, 4, 128, device="cuda").bfloat16() for _ in range(2))
        to = (pos, slots, kc, vc, cos_sin)
        if fused:
            q = ops.step_linear_rope_and_cache(x, w, 8, *to)
        else:
            y16 = ops.step_linear(x, w).view(m, 16, 128)
            q = ops.rope_and_cache(y16[:, :8], y16[:, 8:12], y16[:, 12:], *to)[0]
        both.append([t.double() for t in (q, kc, vc)])
    dy = dy.view(m, 16, 128)
    # a rotated value has both of its pair, each times at most 1
    pair = dy + dy.roll(64, -1)
    for a, b, d in zip(*both, (pair[:, :8], pair[:, 8:12], dy[:, 12:])):
        assert ((a - b).abs() <= d + ulp * b.abs()).all()
