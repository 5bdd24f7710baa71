"""Conv2D layers of one tap, unit stride and no padding, which run as products of matrices: images and channels at the edges of
pieces, slabs and tiles, one and many samples, layers large enough for the streaming kernel and for two separate gradients;
against float64 products."""
import pytest
import torch

import helpers as hp
from test_gpu_conv_any import rel, tensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# fp32: sums of at most 3e4 products in slabs of 32, sqrt(32 / 3) and sqrt(1e3 / 3) roundings of 2^-25 on either side of the
# slabs; fp16: the result's own rounding, 2^-11 at most
TOL = {"fp32": 2e-6, "fp16": 5e-4}

CASES = [  # samples, Ci, Co, pixels (rows, columns)
    (1, 8, 9, 1, 7), (1, 8, 8, 2, 4), (3, 65, 9, 3, 3), (40, 9, 33, 5, 13), (2, 300, 70, 8, 8), (7, 16, 130, 10, 13),
    (30, 24, 40, 23, 25),                      # columns enough for the streaming kernel
    (20, 65, 130, 31, 33), (1, 129, 8, 64, 65),
    (70, 100, 160, 37, 32)]                    # fp32 above 40 MB


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("hwc", [0, 1])
@pytest.mark.parametrize("bias", [0, 1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_layer(pkg, gpu, dt, hwc, bias, case):
    ns, Ci, Co, H, W = case
    P = H * W
    g = torch.Generator(device=DEV).manual_seed(Ci * Co + H)
    act = (lambda c: (ns, H, W, c)) if hwc else (lambda c: (ns, c, H, W))
    x, dx, dy, y = tensor(g, act(Ci), dt), tensor(g, act(Ci), dt), tensor(g, act(Co), dt), tensor(g, act(Co), dt)
    w, dw = tensor(g, (Co, Ci), dt), tensor(g, (Co, Ci), dt)
    b, db = (tensor(g, (Co,), dt), tensor(g, (Co,), dt)) if bias else (None, None)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, Ci, H, W, Co, 1, 1, H, W, (0, 0, 0, 0), (1, 1), hwc, bias=b, dbias=db)
    pkg.call("ptl_conv2d_%s_fw_batched" % dt, a, ns)
    pkg.call("ptl_conv2d_%s_bw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    rows = (lambda t, c: t.double().reshape(ns * P, c)) if hwc else (lambda t, c: t.double().reshape(ns, c, P).permute(0, 2, 1).reshape(ns * P, c))
    X, D, Wd = rows(x, Ci), rows(dy, Co), w.double()
    assert rel(rows(y, Co), X @ Wd.t() + (b.double() if bias else 0)) <= TOL[dt]
    assert rel(rows(dx, Ci), D @ Wd) <= TOL[dt]
    assert rel(dw, D.t() @ X) <= TOL[dt]
    if bias:
        assert rel(db, D.sum(0)) <= TOL[dt]


@pytest.mark.parametrize("dt,hwc,bias,ns,Ci,Co,H,W", [
    ("fp32", 0, 0, 120, 33, 256, 25, 25), ("fp32", 0, 1, 30, 128, 260, 25, 25), ("fp32", 0, 1, 30, 128, 255, 25, 25), ("fp32", 0, 1, 120, 32, 256, 25, 25),
    ("fp32", 0, 1, 90, 132, 32, 41, 37), ("fp32", 0, 0, 90, 132, 33, 41, 37), ("fp32", 0, 1, 60, 129, 128, 32, 32), ("fp32", 0, 1, 60, 129, 128, 33, 32),
    ("fp32", 0, 0, 512, 65, 64, 6, 8), ("fp32", 0, 1, 260, 20, 70, 1, 15), ("fp32", 0, 0, 511, 65, 64, 7, 7),  # images of 48 pixels
    ("fp32", 1, 0, 9, 8, 20, 41, 37), ("fp32", 1, 0, 9, 16, 64, 41, 37), ("fp32", 1, 0, 9, 20, 64, 41, 37), ("fp32", 1, 0, 9, 12, 66, 41, 37),
    ("fp32", 1, 0, 600, 16, 32, 72, 72),                                                                         # 3.2 GFLOP
    ("fp16", 1, 1, 33, 24, 32, 64, 64), ("fp16", 1, 1, 32, 9, 17, 64, 64), ("fp16", 1, 1, 31, 24, 32, 64, 64), ("fp16", 1, 1, 33, 24, 33, 64, 64)])
def test_forward_on_both_sides_of_the_lines(pkg, gpu, dt, hwc, bias, ns, Ci, Co, H, W):
    g = torch.Generator(device=DEV).manual_seed(Ci + Co)
    act = (lambda c: (ns, H, W, c)) if hwc else (lambda c: (ns, c, H, W))
    x, y, w, b = tensor(g, act(Ci), dt), tensor(g, act(Co), dt), tensor(g, (Co, Ci), dt), tensor(g, (Co,), dt)
    a, keep = hp.conv2d_args(pkg, x, x, w, w, y, y, Ci, H, W, Co, 1, 1, H, W, (0, 0, 0, 0), (1, 1), hwc, bias=b if bias else None)
    pkg.call("ptl_conv2d_%s_fw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    rows = (lambda t, c: t.double().reshape(-1, c)) if hwc else (lambda t, c: t.double().reshape(ns, c, H * W).permute(0, 2, 1).reshape(-1, c))
    assert rel(rows(y, Co), rows(x, Ci) @ w.double().t() + (b.double() if bias else 0)) <= TOL[dt]
