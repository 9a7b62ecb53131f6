"""Which sizes the kernel of a small decode step's projections takes: those at which it was
measured to be faster than the GEMM library."""
import pytest

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
