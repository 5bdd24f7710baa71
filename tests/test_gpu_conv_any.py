"""Convolutions of any geometry as products with implicit patch matrices: channel counts, images and strides at the edges of
pieces, slabs and tiles, against float64 patch matrices."""
import pytest
import torch
import torch.nn.functional as F

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {"fp32": 3e-6, "fp16": 1e-3}


def tensor(g, shape, dt):
    """Uniform values one element into a buffer whose other elements are NaN: nothing outside may be used."""
    tdt = torch.float32 if dt == "fp32" else torch.float16
    n = 1
    for s in shape:
        n *= s
    buf = torch.full((n + 65,), float("nan"), dtype=tdt, device=DEV)
    t = buf[1:1 + n].view(shape)
    t.copy_(torch.rand(shape, generator=g, device=DEV) * 2 - 1)
    return t


def rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


CASES = [  # batch, Ci, Co, H, W, kernel, stride, padding
    (2, 8, 8, 8, 8, 3, 1, 1), (3, 9, 17, 11, 13, 3, 2, 1), (5, 24, 45, 15, 14, 5, 2, 2), (1, 65, 33, 7, 9, 3, 1, 0),
    (4, 7, 70, 9, 5, 3, 2, 0), (2, 40, 130, 10, 12, 5, 1, 2), (33, 8, 9, 5, 4, 3, 1, 1), (2, 19, 12, 13, 7, 1, 2, 0),
    (3, 130, 129, 9, 9, 3, 1, 1), (1, 16, 8, 40, 3, 3, 1, 1), (2, 12, 20, 6, 6, 4, 2, 1), (2, 10, 11, 12, 12, 2, 2, 0),
    (70, 33, 12, 7, 7, 3, 2, 1), (1, 300, 16, 6, 6, 3, 1, 1)]


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("hwc", [0, 1])
@pytest.mark.parametrize("bias", [0, 1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_convolution(pkg, gpu, dt, hwc, bias, case):
    ns, Ci, Co, H, W, k, s, p = case
    if s == 2 and (H + 2 * p - k) % 2:
        H += 1  # (strides that divide the extent)
    if s == 2 and (W + 2 * p - k) % 2:
        W += 1
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci * Co + H)
    act = (lambda c, h, w: (ns, h, w, c)) if hwc else (lambda c, h, w: (ns, c, h, w))
    wsh = (Co, k, k, Ci) if hwc else (Co, Ci, k, k)
    x, dx, dy, y = tensor(g, act(Ci, H, W), dt), tensor(g, act(Ci, H, W), dt), tensor(g, act(Co, Ho, Wo), dt), tensor(g, act(Co, Ho, Wo), dt)
    w, dw = tensor(g, wsh, dt), tensor(g, wsh, dt)
    b, db = (tensor(g, (Co,), dt), tensor(g, (Co,), dt)) if bias else (None, None)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, Ci, H, W, Co, k, k, Ho, Wo, pad=(p, p, p, p), stride=(s, s), hwc=hwc, bias=b, dbias=db)
    gpu.ptl_set_gemm_path(7)
    try:
        pkg.call("ptl_conv2d_%s_fw_batched" % dt, a, ns)
        pkg.call("ptl_conv2d_%s_bw_batched" % dt, a, ns)
        assert gpu.ptl_sync() == 0
    finally:
        gpu.ptl_set_gemm_path(0)
    chw = (lambda t: t.double().permute(0, 3, 1, 2)) if hwc else (lambda t: t.double())
    cols = F.unfold(chw(x), k, padding=p, stride=s)  # [ns][Ci k k][P]
    Wm, D = chw(w).reshape(Co, -1), chw(dy).reshape(ns, Co, -1)
    ref_y = (Wm @ cols).view(ns, Co, Ho, Wo) + (b.double().view(1, Co, 1, 1) if bias else 0)
    ref_dw = (D.permute(1, 0, 2).reshape(Co, -1) @ cols.permute(0, 2, 1).reshape(-1, Ci * k * k)).view(Co, Ci, k, k)
    ref_dx = F.fold(Wm.t() @ D, (H, W), k, padding=p, stride=s)
    assert rel(chw(y), ref_y) <= TOL[dt]
    assert rel(chw(dw), ref_dw) <= TOL[dt]
    assert rel(chw(dx), ref_dx) <= TOL[dt]
    if bias:
        assert rel(db, D.sum((0, 2))) <= TOL[dt]


# (channel-major fp16 layers without a bias: at 30 tiles of 64 x 64 and 550 terms the gathering product takes them)
@pytest.mark.parametrize("ns,Ci,Co,H,k,s,p", [(4, 62, 65, 15, 3, 1, 1), (4, 61, 65, 15, 3, 1, 1), (4, 62, 32, 15, 3, 1, 1), (4, 62, 33, 15, 3, 1, 1),
                                              (3, 64, 160, 25, 3, 1, 1), (2, 40, 130, 25, 5, 2, 2), (1, 512, 156, 5, 5, 2, 2), (8, 62, 256, 11, 3, 1, 1)])
def test_forward_on_few_tiles(pkg, gpu, ns, Ci, Co, H, k, s, p):
    Ho = (H + 2 * p - k) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci * Co + H)
    x, y, w = (tensor(g, sh, "fp16") for sh in ((ns, Ci, H, H), (ns, Co, Ho, Ho), (Co, Ci, k, k)))
    a, keep = hp.conv2d_args(pkg, x, x, w, w, y, y, Ci, H, H, Co, k, k, Ho, Ho, pad=(p,) * 4, stride=(s, s))
    pkg.call("ptl_conv2d_fp16_fw_batched", a, ns)
    assert gpu.ptl_sync() == 0
    ref = w.double().reshape(Co, -1) @ F.unfold(x.double(), k, padding=p, stride=s)
    assert rel(y.double().reshape(ns, Co, -1), ref) <= TOL["fp16"]
