"""Which sizes the kernel of a small decode step's projections takes: those at which it was
measured to be faster than the GEMM library."""
import pytest
import torch

from agentcontrolplane_amd import ops


@pytest.mark.parametrize("m,outs,k,glu,pays", [
    # where the library was 4 to 50% faster
    (1, 65536, 1024, False, False), (4, 128256, 256, False, False), (1, 16, 5120, False, False),
    (1, 512, 14336, False, False), (4, 128, 6144, False, False), (4, 4608, 4608, False, False),
    (4, 5120, 4608, False, False), (1, 5120, 7168, False, False), (4, 6144, 5120, False, False),
    (4, 6144, 7168, False, False), (4, 6144, 8192, False, False), (1, 1024, 7168, True, False),
    (4, 2048, 7168, True, False), (4, 2048, 8192, True, False), (1, 2048, 14336, True, False),
    (4, 5632, 14336, True, False), (5, 4096, 4096, False, False),
    # where this kernel was 3 to 200% faster
    (1, 2048, 64, False, True), (4, 16, 4096, False, True), (4, 4608, 3584, False, True),
    (1, 4096, 4096, False, True), (4, 6144, 4096, False, True), (1, 128256, 4096, False, True),
    (4, 20048, 2048, False, True), (4, 65536, 1536, False, True), (4, 1024, 4608, False, True),
    (1, 6144, 5120, False, True), (4, 15360, 5120, False, True), (4, 32000, 5120, False, True),
    (4, 2048, 6144, False, True), (1, 4096, 7168, False, True), (4, 1024, 8064, False, True),
    (4, 6144, 8064, False, True), (4, 4096, 14336, False, True), (1, 6144, 14336, False, True),
    (4, 5632, 2048, True, True), (4, 18944, 3584, True, True), (4, 14336, 4096, True, True),
    (1, 256, 5120, True, True), (4, 2048, 6144, True, True), (4, 2048, 8064, True, True),
    (4, 2048, 11008, True, True), (4, 4096, 14336, True, True),
])
def test_few_rows_go_where_they_are_faster(m, outs, k, glu, pays):
    assert ops._few_rows_pay(m, outs, k, glu) == pays


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 3, 4])
@pytest.mark.parametrize("n,k", [(2056, 5664), (6160, 3104)])
def test_step_linear_of_whole_lines(m, n, k):
    """Outputs that are no whole tiles and half a line at the end, against double precision."""
    x, w = torch.randn(m, k).bfloat16().cuda(), torch.randn(n, k).bfloat16().cuda()
    assert ops._few_rows(x, w)
    got, want = ops.step_linear(x, w).double(), x.double() @ w.double().T
    slack = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + slack + 1e-30).all()
