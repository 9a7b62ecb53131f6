"""Products of many rows (csrc/linear.hip): every tile at its edges against double precision,
and which calls its rule takes."""
import pytest
import torch

from agentcontrolplane_amd import ops
from agentcontrolplane_amd.engine.config import ClampedGluSpec

TILES = range(13)


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
    beside the outputs.  The last case has several tiles a workgroup."""
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
    form = (7.0, 1.702, 1.0, 0.0) if unit == "glu" else (0.0,) * 4
    got = hip.linear(x, w, None, unit, form, tile=tile, splits=splits).double()
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
    assert ((got - want).abs() <= bound + 2.0 ** -7 * want.abs() + 1e-30).all()


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


def test_rule_of_many_rows():
    """Few rows and small weights stay where they were; so does what the library is faster at."""
    pay = ops._many_rows_pay
    assert not pay(4, 4096, 4096, False) and pay(5, 4096, 4096, False)
    assert not pay(64, 2048, 64, False)
    assert not pay(8192, 4096, 4096, False) and pay(8192, 8192, 4096, True)
    assert pay(10000, 4096, 4096, False) and pay(16000, 4096, 14336, False)
    # not on the CPU
    x, w = torch.zeros(64, 1024).bfloat16(), torch.zeros(2048, 1024).bfloat16()
    assert not ops._many_rows(x, w)
    out = torch.empty(64, 1024).bfloat16()
    ops.step_linear_glu(x + 1, w + 0.01, ClampedGluSpec(1024, 7.0, 1.702, 1.0), out)
    want = torch.empty_like(out)
    ops.clamped_glu(ops.linear(x + 1, w + 0.01), 7.0, 1.702, 1.0, want)
    assert torch.equal(out, want)
