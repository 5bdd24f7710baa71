"""Sizes whose launches would have 2^32 threads and more along one axis."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,m", [(2 ** 30 + 67, 1), (2 ** 29 + 3, 2), (1, 2 ** 29 + 5)])
def test_transposition_of_a_long_matrix(pkg, gpu, n, m):
    x = torch.arange(n * m, device=DEV, dtype=torch.int32).to(torch.int16).view(torch.float16).view(n, m)
    out = torch.zeros(m, n, device=DEV, dtype=torch.float16)
    a = pkg.TranspArgs()
    a.in_matrix, a.out_matrix, a.N, a.M = pkg.addr(x), pkg.addr(out), n, m
    pkg.call("transpose_matrix_fp16", a)
    assert gpu.ptl_sync() == 0
    assert torch.equal(out.view(torch.int16), x.t().contiguous().view(torch.int16))
