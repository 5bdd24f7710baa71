"""Patch matrices whose rows are no whole 16-byte chunks, start anywhere and are built in pieces of the channels, and
transpositions of any alignment: bit for bit."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def shifted(t, n):
    """t, n elements into a buffer of its own."""
    buf = torch.full((t.numel() + n + 16,), 5.0, dtype=t.dtype, device=DEV)
    v = buf[n:n + t.numel()].view(t.shape)
    v.copy_(t)
    return v, buf


@pytest.mark.parametrize("dt,tdt", [("fp16", torch.float16), ("fp32", torch.float32)])
@pytest.mark.parametrize("C,H,W,K,pad,stride,shift", [(83, 9, 21, 3, 1, 1, 0), (163, 5, 17, 3, 1, 1, 1), (9, 6, 16, 1, 0, 1, 3),
                                                     (1, 40, 33, 3, 1, 1, 0), (241, 4, 19, 5, 2, 1, 1), (31, 9, 37, 3, 1, 2, 0),
                                                     (65, 300, 18, 3, 0, 1, 0)])
def test_im2row(pkg, gpu, dt, tdt, C, H, W, K, pad, stride, shift):
    x, _ = shifted(torch.rand(C, H, W, device=DEV).to(tdt), shift)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    out, buf = shifted(torch.zeros(Ho * Wo, C * K * K, device=DEV, dtype=tdt), shift)
    a = pkg.Im2colArgs()
    keep = [pkg.blob(x, None, C, H, W), pkg.blob(None, None, C, K, K), pkg.blob(None, None, 4, Ho, Wo)]
    a.input, a.c, a.output = [pkg.structs.C.pointer(b) for b in keep]
    a.pBuffer = pkg.addr(out)
    a.Lpad = a.Rpad = a.Upad = a.Dpad = pad
    a.stride_h = a.stride_w = stride
    pkg.call("pulp_im2row_" + dt, a)
    assert gpu.ptl_sync() == 0
    ref = F.unfold(x.float()[None], K, padding=pad, stride=stride)[0].t().to(tdt)
    assert torch.equal(out, ref)
    assert bool((buf[:shift] == 5).all()) and bool((buf[shift + out.numel():] == 5).all())


@pytest.mark.parametrize("half,tdt", [("_fp16", torch.float16), ("", torch.float32)])
@pytest.mark.parametrize("N,M,shift", [(64, 64, 1), (65, 63, 0), (7, 200, 3), (200, 7, 1), (1, 9, 0), (129, 257, 1)])
def test_transposition(pkg, gpu, half, tdt, N, M, shift):
    x, _ = shifted(torch.rand(N, M, device=DEV).to(tdt), shift)
    out, buf = shifted(torch.zeros(M, N, device=DEV, dtype=tdt), shift)
    a = pkg.TranspArgs()
    a.in_matrix, a.out_matrix, a.N, a.M = pkg.addr(x), pkg.addr(out), N, M
    pkg.call("transpose_matrix" + half, a)
    assert gpu.ptl_sync() == 0
    assert torch.equal(out, x.t())
    assert bool((buf[:shift] == 5).all()) and bool((buf[shift + out.numel():] == 5).all())
