"""Patch matrices of tensors whose rows are pieces from any place, block transpositions in small tiles, transpositions with
tiles in runs: bit for bit at the edges of pieces and tiles."""
import pytest
import torch
import torch.nn.functional as F

from test_gpu_patch_rows import DEV, shifted

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dt,tdt", [("fp16", torch.float16), ("fp32", torch.float32)])


@BOTH
@pytest.mark.parametrize("H,W,K,pad,stride", [(3, 7, 3, 9, 1), (5, 8, 3, 8, 1), (9, 9, 3, 1, 1), (7, 35, 5, 17, 1), (2, 41, 3, 1, 1),
                                              (9, 67, 1, 0, 2), (21, 131, 3, 1, 1), (6, 3, 3, 9, 1)])
@pytest.mark.parametrize("C", [9, 71])
def test_im2row(pkg, gpu, dt, tdt, C, H, W, K, pad, stride):
    x, _ = shifted(torch.rand(C, H, W, device=DEV).to(tdt), 1)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    out, buf = shifted(torch.zeros(Ho * Wo, C * K * K, device=DEV, dtype=tdt), 1)
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
    assert bool((buf[:1] == 5).all()) and bool((buf[1 + out.numel():] == 5).all())


@BOTH
@pytest.mark.parametrize("Ci,Co,K,shift", [(71, 65, 1, 0), (8, 521, 1, 1), (9, 65, 3, 0), (57, 9, 3, 1), (33, 31, 3, 1), (9, 23, 5, 0),
                                           (150, 163, 3, 0), (510, 515, 3, 1)])
def test_blocktranspose(pkg, gpu, dt, tdt, Ci, Co, K, shift):
    w, _ = shifted(torch.rand(Co, Ci, K * K, device=DEV).to(tdt), shift)
    out, buf = shifted(torch.zeros(Ci, Co, K * K, device=DEV, dtype=tdt), shift)
    a = pkg.BlocktranspArgs()
    a.weights, a.bt_weights, a.Cin, a.Cout, a.Hk, a.Wk, a.HWC = pkg.addr(w), pkg.addr(out), Ci, Co, K, K, 0
    pkg.call("pulp_blocktransp_" + dt, a)
    assert gpu.ptl_sync() == 0
    assert torch.equal(out, w.flip(2).permute(1, 0, 2))
    assert bool((buf[:shift] == 5).all()) and bool((buf[shift + out.numel():] == 5).all())


@pytest.mark.parametrize("N,M", [(1, 1), (64 * 3, 64 * 5), (64 * 3 + 1, 64 * 5 + 1), (449, 64), (64, 513), (577, 65)])
def test_transposition(pkg, gpu, N, M):
    x, _ = shifted(torch.rand(N, M, device=DEV), 1)
    out, buf = shifted(torch.zeros(M, N, device=DEV), 1)
    a = pkg.TranspArgs()
    a.in_matrix, a.out_matrix, a.N, a.M = pkg.addr(x), pkg.addr(out), N, M
    pkg.call("transpose_matrix", a)
    assert gpu.ptl_sync() == 0
    assert torch.equal(out, x.t())
    assert bool((buf[:1] == 5).all()) and bool((buf[1 + out.numel():] == 5).all())
