"""Sizes whose launches would have 2^32 threads and more along one axis."""
import pytest
import torch

import helpers as hp

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


@pytest.mark.parametrize("ns,path", [(66, 0), (64, 8), (66, 8)])
def test_one_channel_over_many_pixels(pkg, gpu, ns, path):
    """3 x 3, one channel to one: 8.38 and 8.64 million tiles of the input gradient; 8.39 million workgroups of 512 threads are 2^32."""
    H, W = 2900, 2890
    g = torch.Generator(device=DEV).manual_seed(1)
    dy = torch.randint(-2, 3, (ns, H, W), generator=g, device=DEV, dtype=torch.int8).half()
    x, dx, dw = torch.zeros_like(dy), torch.full_like(dy, 7), torch.zeros(9, device=DEV).half()
    w = torch.arange(1, 10, device=DEV).half()
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, dy, dy, 1, H, W, 1, 3, 3, H, W, pad=(1, 1, 1, 1))
    gpu.ptl_set_gemm_path(path)
    try:
        pkg.call("ptl_conv2d_fp16_bw_batched", a, ns)
    finally:
        gpu.ptl_set_gemm_path(0)
    assert gpu.ptl_sync() == 0
    for b in (0, ns // 2, ns - 1):
        ref = torch.nn.functional.unfold(dy[b].float().view(1, 1, H, W), 3, padding=1)[0].t() @ w.float().flip(0)
        assert torch.equal(dx[b], ref.view(H, W).half())
