"""3x3 depthwise layers whose planes are no whole number of the kernels' blocks (7 rows x 16 bytes of columns), start
anywhere, have any padding, or are smaller than one block, against fp32 convolutions."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def placed(t, n):
    """t, n elements into a buffer whose end is the tensor's."""
    buf = torch.full((t.numel() + n,), float("nan"), dtype=t.dtype, device=DEV)
    v = buf[n:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("b,C,H,W,pad,shift", [(1, 1, 3, 14, 0, 0), (2, 3, 6, 9, 1, 1), (3, 5, 9, 9, 0, 1), (1, 7, 9, 12, 1, 0),
                                              (5, 2, 16, 33, 2, 3), (2, 9, 15, 58, 0, 0), (3, 2, 4, 5, 1, 1), (37, 17, 30, 31, 1, 0),
                                              (1, 16, 58, 113, 0, 1), (2, 2, 5, 4, 3, 1),
                                              # the blocks of a plane in shares, the last one short
                                              (1, 3, 230, 131, 1, 1), (1, 2, 301, 299, 0, 1), (2, 3, 60, 150, 1, 3), (5, 1, 257, 129, 2, 0)])
def test_depthwise_blocks(pkg, gpu, dt, b, C, H, W, pad, shift):
    tdt = torch.float32 if dt == "fp32" else torch.float16
    Ho, Wo = H + 2 * pad - 2, W + 2 * pad - 2
    x = placed(torch.rand(b, C, H, W, device=DEV).to(tdt) - 0.5, shift)
    w = placed(torch.rand(C, 3, 3, device=DEV).to(tdt) - 0.5, shift)
    dy = placed(torch.rand(b, C, Ho, Wo, device=DEV).to(tdt) - 0.5, shift)
    y, dx, dw = (placed(torch.zeros_like(t), shift) for t in (dy, x, w))
    a = pkg.DepthWiseConvArgs() if dt == "fp32" else pkg.DepthWiseConvArgsFp16()
    keep = [pkg.blob(x, dx, C, H, W), pkg.blob(w, dw, 1, 3, 3, C * 9), pkg.blob(y, dy, C, Ho, Wo)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(k) for k in keep]
    a.Lpad = a.Rpad = a.Upad = a.Dpad = pad
    if dt == "fp32":
        a.stride_h = a.stride_w = 1
    if b == 1:
        for step in ("fw", "bw"):
            pkg.call("pulp_conv_dw_%s_%s_cl" % (dt, step), a)
    else:
        for step in ("fw", "wg", "ig"):
            pkg.call("ptl_conv_dw_%s_%s_batched" % (dt, step), a, b)
    assert gpu.ptl_sync() == 0
    # (in 64 bits: a weight gradient of 89 000 products in the CPU's 32 has been 1.0e-5 of the largest off by itself)
    xr, wr = x.double().cpu().requires_grad_(), w.double().cpu()[:, None].requires_grad_()
    yr = F.conv2d(xr, wr, padding=pad, groups=C)
    yr.backward(dy.double().cpu())
    for got, want in ((y, yr.detach()), (dx, xr.grad), (dw, wr.grad[:, 0])):
        scale = float(want.abs().max()) + 1e-3
        assert float((got.double().cpu() - want).abs().max()) <= (2e-3 if dt == "fp16" else 1e-5) * scale


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
# rows and columns of the gradient that end inside a block; several planes; the blocks of a plane in shares
@pytest.mark.parametrize("b,C,H,W", [(1, 3, 20, 31), (2, 2, 34, 35), (4, 5, 12, 45), (1, 2, 301, 299)])
def test_infinities_in_the_last_rows_and_columns(pkg, gpu, dt, b, C, H, W):
    """An infinity of the input reaches the taps that a gradient meets it with and no other: of the last row and column (no
    padding) only one tap."""
    tdt = torch.float32 if dt == "fp32" else torch.float16
    x, w = (torch.rand(s, device=DEV).to(tdt) for s in ((b, C, H, W), (C, 3, 3)))
    dy = (torch.rand(b, C, H - 2, W - 2, device=DEV) + 0.5).to(tdt)
    inf = float("inf")
    x[0, 0, H - 1, W - 1] = inf      # tap (2, 2)
    x[b - 1, 1, H - 1, 0] = -inf     # tap (2, 0)
    dw = torch.zeros_like(w)
    a = pkg.DepthWiseConvArgs() if dt == "fp32" else pkg.DepthWiseConvArgsFp16()
    y, dx = torch.zeros_like(dy), torch.zeros_like(x)
    keep = [pkg.blob(x, dx, C, H, W), pkg.blob(w, dw, 1, 3, 3, C * 9), pkg.blob(y, dy, C, H - 2, W - 2)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(k) for k in keep]
    a.Lpad = a.Rpad = a.Upad = a.Dpad = 0
    if dt == "fp32":
        a.stride_h = a.stride_w = 1
    pkg.call("ptl_conv_dw_%s_wg_batched" % dt, a, b)
    assert gpu.ptl_sync() == 0
    X, D = x.double(), dy.double()
    want = torch.stack([torch.stack([(X[:, :, i:i + H - 2, j:j + W - 2] * D).sum((0, 2, 3)) for j in range(3)], 1) for i in range(3)], 1)
    finite = want.isfinite()
    assert int((~finite).sum()) == 2 and float(want[0, 2, 2]) == inf and float(want[1, 2, 0]) == -inf
    assert bool((dw.double()[~finite] == want[~finite]).all())
    err = (dw.double() - want)[finite].norm() / want[finite].norm()
    assert float(err) <= (1e-3 if dt == "fp16" else 1e-6)
