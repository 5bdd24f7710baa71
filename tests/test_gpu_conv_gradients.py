"""Both gradients of a convolution in one launch: filters read in place (channel-major: element by element, channel-minor: in
pieces whose last one reaches over the end), phases of strided layers that no tap reaches, split contractions with bias
gradients, and the input gradient alone; against float64 patch matrices."""
import pytest
import torch
import torch.nn.functional as F

import helpers as hp
from test_gpu_conv_any import rel, tensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# fp32: a chain of 3e4 rounded additions, sqrt(n / 3) * 2^-25 (sums of slabs are shorter); fp16: the result's rounding, 2^-11
TOL = {"fp32": 3e-6, "fp16": 5e-4}

CASES = [  # batch, Ci, Co, H, W, kernel, stride, padding
    (1, 8, 8, 7, 9, 3, 1, 1),        # one workgroup a product, slabs not full
    (2, 65, 9, 8, 8, 3, 1, 1),       # input channels one over a tile
    (3, 17, 70, 11, 12, 3, 1, 0),    # output channels in pieces with a remainder, several tiles
    (40, 9, 33, 13, 13, 5, 1, 2),    # 25 taps, weight gradient cut many times
    (2, 300, 12, 6, 6, 3, 1, 1),     # five tiles of input channels
    (5, 24, 45, 15, 14, 5, 2, 2),    # four phases of 9, 6, 6 and 4 taps
    (2, 20, 130, 10, 12, 1, 2, 0),   # three phases without a tap
    (3, 12, 20, 7, 7, 3, 2, 1),
    (2, 640, 24, 5, 5, 3, 1, 1)]     # input gradient's contraction short, weight gradient's wide


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("hwc,path", [(0, 8), (0, 9), (1, 8)])  # (channel-minor tensors are never copied)
@pytest.mark.parametrize("bias", [0, 1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gradients(pkg, gpu, dt, hwc, path, bias, case):
    ns, Ci, Co, H, W, k, s, p = case
    H, W = H + (H + 2 * p - k) % s, W + (W + 2 * p - k) % s
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci * Co + H)
    act = (lambda c, h, w: (ns, h, w, c)) if hwc else (lambda c, h, w: (ns, c, h, w))
    wsh = (Co, k, k, Ci) if hwc else (Co, Ci, k, k)
    x, dx, dy = tensor(g, act(Ci, H, W), dt), tensor(g, act(Ci, H, W), dt), tensor(g, act(Co, Ho, Wo), dt)
    w, dw = tensor(g, wsh, dt), tensor(g, wsh, dt)
    b, db = (tensor(g, (Co,), dt), tensor(g, (Co,), dt)) if bias else (None, None)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, dy, dy, Ci, H, W, Co, k, k, Ho, Wo, pad=(p, p, p, p), stride=(s, s), hwc=hwc, bias=b, dbias=db)
    chw = (lambda t: t.double().permute(0, 3, 1, 2)) if hwc else (lambda t: t.double())
    cols = F.unfold(chw(x), k, padding=p, stride=s)
    Wm, D = chw(w).reshape(Co, -1), chw(dy).reshape(ns, Co, -1)
    ref_dw = (D.permute(1, 0, 2).reshape(Co, -1) @ cols.permute(0, 2, 1).reshape(-1, Ci * k * k)).view(Co, Ci, k, k)
    ref_dx = F.fold(Wm.t() @ D, (H, W), k, padding=p, stride=s)
    gpu.ptl_set_gemm_path(path)
    try:
        for step in ("bw", "ig"):
            dx.fill_(7)
            pkg.call("ptl_conv2d_%s_%s_batched" % (dt, step), a, ns)
            assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_tile() == 64064
            assert gpu.ptl_last_conv_resident() == (4 if path == 9 else 0)
            assert rel(chw(dx), ref_dx) <= TOL[dt], step
    finally:
        gpu.ptl_set_gemm_path(0)
    assert rel(chw(dw), ref_dw) <= TOL[dt]
    if bias:
        assert rel(db, D.sum((0, 2))) <= TOL[dt]


@pytest.mark.parametrize("dt,hwc,bias,ns,Ci,Co,H,W,k,s", [
    ("fp32", 0, 1, 82, 128, 63, 32, 32, 1, 1), ("fp32", 0, 0, 81, 128, 63, 32, 32, 1, 1), ("fp32", 0, 0, 83, 128, 64, 32, 32, 1, 1),  # 64 MB
    ("fp32", 1, 1, 82, 128, 63, 32, 32, 1, 1), ("fp32", 1, 0, 83, 127, 63, 32, 32, 1, 1),
    ("fp16", 1, 0, 32, 24, 32, 63, 63, 1, 2), ("fp16", 1, 1, 33, 9, 96, 63, 63, 1, 2), ("fp16", 1, 0, 31, 24, 32, 63, 63, 1, 2),  # 32768 pixels
    ("fp32", 1, 0, 82, 16, 32, 63, 63, 1, 2), ("fp32", 1, 0, 85, 16, 32, 63, 63, 1, 2), ("fp32", 1, 1, 85, 16, 32, 63, 63, 1, 2),  # 32 MB
    ("fp16", 0, 0, 15, 9, 7, 64, 64, 3, 1), ("fp16", 0, 1, 15, 16, 16, 64, 64, 3, 1), ("fp16", 0, 1, 14, 16, 16, 64, 64, 3, 1)])  # 60000
def test_gradients_on_both_sides_of_the_lines_to_single_steps(pkg, gpu, dt, hwc, bias, ns, Ci, Co, H, W, k, s):
    p, Ho, Wo = k // 2, (H - 1) // s + 1, (W - 1) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci * Co + ns)
    act = (lambda c, h, w: (ns, h, w, c)) if hwc else (lambda c, h, w: (ns, c, h, w))
    x, dx, dy = tensor(g, act(Ci, H, W), dt), tensor(g, act(Ci, H, W), dt), tensor(g, act(Co, Ho, Wo), dt)
    w, dw = (tensor(g, (Co, k, k, Ci) if hwc else (Co, Ci, k, k), dt) for _ in range(2))
    b, db = (tensor(g, (Co,), dt), tensor(g, (Co,), dt)) if bias else (None, None)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, dy, dy, Ci, H, W, Co, k, k, Ho, Wo, pad=(p, p, p, p), stride=(s, s), hwc=hwc, bias=b, dbias=db)
    pkg.call("ptl_conv2d_%s_bw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    chw = (lambda t: t.double().permute(0, 3, 1, 2)) if hwc else (lambda t: t.double())
    cols, D, Wm = F.unfold(chw(x), k, padding=p, stride=s), chw(dy).reshape(ns, Co, -1), chw(w).reshape(Co, -1)
    assert rel(chw(dw).reshape(Co, -1), D.permute(1, 0, 2).reshape(Co, -1) @ cols.permute(0, 2, 1).reshape(-1, Ci * k * k)) <= TOL[dt]
    assert rel(chw(dx), F.fold(Wm.t() @ D, (H, W), k, padding=p, stride=s)) <= TOL[dt]
    if bias:
        assert rel(db, D.sum((0, 2))) <= TOL[dt]
    if k == 3:
        assert gpu.ptl_last_conv_direct() == (ns == 15)
