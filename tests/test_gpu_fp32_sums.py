"""fp32 products of any size: their sums are those of slabs of k added up, not one chain of additions.

A chain of n additions of values of random sign with independent roundings of at most u = 2^-24 leaves a relative error of
u / sqrt(3) * sqrt(n / 2) (the i-th rounds a partial sum of sqrt(i) values); slabs of 32 and a chain of their K / 32 sums
u / sqrt(3) * sqrt((32 + K / 32) / 2), which waves along k and split contractions make smaller."""
import ctypes
import math

import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bound(k):
    return 2.0 ** -24 / math.sqrt(3) * math.sqrt((32 + k / 32) / 2)


def error(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("b,i,o", [(1031, 2049, 1027), (2051, 1029, 1031), (259, 4099, 4097), (67, 4101, 65)])
def test_linear(pkg, gpu, b, i, o):
    r = lambda *s: torch.rand(*s, device=DEV) * 2 - 1
    x, w, dy = r(b, i), r(o, i), r(b, o)
    y, dx, dw = torch.zeros_like(dy), torch.zeros_like(x), torch.zeros_like(w)
    a = pkg.LinearArgs()
    keep = [pkg.blob(x, dx, 1, 1, i), pkg.blob(w, dw, 1, o, i), pkg.blob(y, dy, 1, 1, o)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(k) for k in keep]
    pkg.call("ptl_linear_fp32_fw_batched", a, b)
    pkg.call("ptl_linear_fp32_bw_batched", a, b)
    assert gpu.ptl_sync() == 0
    X, W, G = x.double(), w.double(), dy.double()
    assert error(y, X @ W.t()) <= bound(i)
    assert error(dx, G @ W) <= bound(o)
    assert error(dw, G.t() @ X) <= bound(b)


@pytest.mark.parametrize("b,c,co,h,k,s", [(24, 57, 131, 31, 5, 2), (48, 130, 67, 29, 3, 2), (9, 65, 190, 33, 5, 1)])
@pytest.mark.parametrize("hwc", [0, 1])
def test_conv(pkg, gpu, b, c, co, h, k, s, hwc):
    p, ho = k // 2, (h + 2 * (k // 2) - k) // s + 1
    act = (lambda c, n: (b, n, n, c)) if hwc else (lambda c, n: (b, c, n, n))
    chw = (lambda t: t.permute(0, 3, 1, 2).contiguous()) if hwc else (lambda t: t)
    r = lambda sh: torch.rand(sh, device=DEV) * 2 - 1
    x, dy, w = r(act(c, h)), r(act(co, ho)), r((co, k, k, c) if hwc else (co, c, k, k))
    y, dx, dw = torch.zeros_like(dy), torch.zeros_like(x), torch.zeros_like(w)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, c, h, h, co, k, k, ho, ho, pad=(p, p, p, p), stride=(s, s), hwc=hwc)
    gpu.ptl_set_gemm_path(7)
    assert gpu.ptl_conv2d_fp32_fw_batched(ctypes.byref(a), b) == 0
    assert gpu.ptl_conv2d_fp32_bw_batched(ctypes.byref(a), b) == 0
    gpu.ptl_set_gemm_path(0)
    assert gpu.ptl_sync() == 0
    cols = torch.nn.functional.unfold(chw(x).double(), k, padding=p, stride=s)
    W, G = chw(w).double().reshape(co, -1), chw(dy).double().reshape(b, co, -1)
    assert error(chw(y), torch.matmul(W, cols).view(b, co, ho, ho)) <= bound(c * k * k)
    rw = G.permute(1, 0, 2).reshape(co, -1) @ cols.permute(0, 2, 1).reshape(-1, c * k * k)
    assert error(chw(dw), rw.view(co, c, k, k)) <= bound(b * ho * ho)
    rx = torch.nn.functional.fold(torch.matmul(W.t().contiguous(), G), (h, h), k, padding=p, stride=s)
    assert error(chw(dx), rx) <= bound(co * k * k)


@pytest.mark.parametrize("b,c,h,w", [(3, 5, 67, 45), (40, 16, 33, 29), (200, 3, 18, 23), (1, 2, 513, 511)])
def test_depthwise_weight_gradient(pkg, gpu, b, c, h, w):
    """Rows of four products apart, a lane's rows in a chain of at most all rows over 64 lanes, then trees."""
    r = lambda *s: torch.rand(*s, device=DEV) * 2 - 1
    x, dy = r(b, c, h + 2, w + 2), r(b, c, h, w)
    k, dw = torch.zeros(c, 3, 3, device=DEV), torch.zeros(c, 3, 3, device=DEV)
    a = pkg.DepthWiseConvArgs()
    keep = [pkg.blob(x, None, c, h + 2, w + 2), pkg.blob(k, dw, 1, 3, 3, c * 9), pkg.blob(dy, dy, c, h, w)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(t) for t in keep]
    a.stride_h = a.stride_w = 1
    pkg.call("ptl_conv_dw_fp32_wg_batched", a, b)
    assert gpu.ptl_sync() == 0
    X, G = x.double(), dy.double()
    want = torch.stack([(X[:, :, i:i + h, j:j + w] * G).sum((0, 2, 3)) for i in range(3) for j in range(3)], 1).view(c, 3, 3)
    n = b * h * w
    # four products, a chain of rows in a workgroup of 256 lanes of 4 columns (blocks of seven rows: at least that many), trees
    rows = max(7, n / (4 * 256))
    assert error(dw, want) <= 2.0 ** -24 / math.sqrt(3) * math.sqrt((4 + rows) / 2 + math.log2(n))
