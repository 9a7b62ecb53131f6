"""Which sizes the kernel of a small decode step's projections takes: those at which it was
measured to be faster than the GEMM library."""
import pytest
import torch

from agentcontrolplane_amd import ops


@pytest.mark.parametrize("m,outs,k,glu,pays", [
    # where the library was 3 to 50% faster
    (1, 5120, 5120, False, False), (4, 15360, 5120, False, False), (4, 32000, 5120, False, False),
    (4, 4608, 3584, False, False), (4, 18944, 3584, True, False), (1, 4096, 7168, False, False),
    (1, 128, 6144, False, False), (4, 2048, 5632, False, False), (4, 6144, 4096, False, False),
    (1, 65536, 256, False, False), (1, 16384, 3072, False, False), (1, 16, 5120, False, False),
    (1, 128256, 4096, False, False), (4, 4096, 14336, False, False), (5, 4096, 4096, False, False),
    # where this kernel was 3 to 66% faster
    (1, 6144, 4096, False, True), (4, 4096, 4096, False, True), (4, 12288, 4096, False, True),
    (4, 32000, 4096, False, True), (4, 14336, 4096, True, True), (4, 11008, 4096, True, True),
    (4, 3584, 3584, False, True), (4, 20048, 2048, False, True), (1, 2048, 64, False, True),
    (4, 1024, 4608, False, True), (4, 5632, 2048, True, True), (4, 1024, 8064, False, True),
])
def test_few_rows_go_where_they_are_faster(m, outs, k, glu, pays):
    assert ops._few_rows_pay(m, outs, k, glu) == pays


@pytest.mark.parametrize("m,outs,k,glu,pays", [
    (1, 5120, 5120, False, False), (4, 65536, 1024, False, False), (1, 512, 14336, False, False),
    (4, 5120, 13824, False, False), (5, 4096, 14336, False, False),
    (4, 4096, 14336, False, True), (1, 128256, 4096, False, True), (4, 18944, 3584, True, True),
    (1, 4096, 7168, False, True), (4, 65536, 1536, False, True), (4, 6144, 4096, False, True),
])
def test_whole_lines_pay(m, outs, k, glu, pays):
    assert ops._whole_lines_pay(m, outs, k, glu) == pays


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 3, 4])
@pytest.mark.parametrize("n,k", [(2056, 5664), (6160, 3104)])
def test_step_linear_of_whole_lines(m, n, k):
    """Sizes of the second rule, with outputs that are no whole tiles and half a line at the end,
    against double precision."""
    x, w = torch.randn(m, k).bfloat16().cuda(), torch.randn(n, k).bfloat16().cuda()
    assert not ops._few_rows_pay(m, n, k, False) and ops._few_rows(x, w)
    got, want = ops.step_linear(x, w).double(), x.double() @ w.double().T
    slack = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + slack + 1e-30).all()
