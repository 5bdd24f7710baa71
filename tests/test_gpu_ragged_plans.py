"""The plans that large products and convolutions take - tiles of 64 and 128, channel-minor copies of channel-major tensors
with padded channels, phases of strided layers - at sizes that fill no tile, against float64.  The tiles are those that
the cost tables give for 256 CUs; the query behind each call says that the plan is the one meant."""
import pytest
import torch
import torch.nn.functional as F

import helpers as hp
from test_gpu_conv_any import rel, tensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# Sums of up to 50 000 products of uniform values in fp32: each addition rounds by 2^-24 at most, and the errors of a chain of
# n add up like a random walk, sqrt(n / 3) * 2^-25 of the result at the end: 4e-6 for one chain (the matrix instruction
# has several).  fp16: the result's own rounding, 2^-11 at most.
TOL = {"fp32": 4e-6, "fp16": 5e-4}
S, M, L = 32064, 64064, 128128
TALL = 64032

# type, channel-minor, (samples, Ci, Co, H, W, kernel, stride), then (tile, on channel-minor copies) of forward, weight
# gradient, input gradient, and of the input gradient in a call for both
CONV = [
    ("fp32", 0, (9, 200, 300, 14, 14, 3, 1), (M, 0), (M, 1), (M, 0), (L, 1)),
    ("fp32", 0, (8, 500, 500, 14, 14, 3, 1), (M, 0), (L, 1), (M, 0), (L, 1)),
    ("fp32", 0, (64, 40, 300, 21, 21, 3, 1), (M, 0), (L, 0), (M, 0), (M, 0)),
    ("fp32", 0, (128, 100, 70, 21, 21, 3, 2), (S, 0), (S, 0), (L, 0), (L, 0)),
    ("fp32", 1, (64, 130, 129, 28, 28, 3, 1), (L, 0), (L, 0), (L, 0), (L, 0)),
    ("fp32", 1, (128, 100, 70, 21, 21, 3, 2), (TALL, 0), (L, 0), (L, 0), (L, 0)),
    ("fp16", 0, (64, 130, 129, 28, 28, 3, 1), (L, 1), (M, 1), (L, 1), (L, 1)),
    ("fp16", 0, (64, 60, 70, 28, 28, 3, 1), (L, 0), (L, 0), (M, 1), (M, 1)),
    ("fp16", 0, (3, 66, 67, 60, 60, 3, 1), (M, 0), (M, 0), (S, 1), (S, 1)),
    ("fp16", 0, (16, 260, 270, 29, 29, 3, 2), (M, 1), (M, 1), (M, 1), (M, 1)),
    ("fp16", 0, (64, 48, 41, 31, 29, 5, 1), (M, 1), (M, 1), (M, 1), (M, 1)),
    ("fp16", 1, (64, 128, 130, 28, 28, 3, 1), (L, 0), (L, 0), (L, 0), (L, 0)),
    ("fp16", 1, (3, 66, 67, 60, 60, 3, 1), (M, 0), (S, 0), (M, 0), (M, 0)),
]


@pytest.mark.parametrize("case", CONV, ids=lambda c: "%s-%d-%s" % (c[0], c[1], "x".join(map(str, c[2]))))
@pytest.mark.parametrize("bias", [0, 1])
def test_convolutions(pkg, gpu, case, bias):
    dt, hwc, (ns, Ci, Co, H, W, k, s), *plans = case
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci * Co + H)
    act = (lambda c, h, w: (ns, h, w, c)) if hwc else (lambda c, h, w: (ns, c, h, w))
    wsh = (Co, k, k, Ci) if hwc else (Co, Ci, k, k)
    x, dx, dy, y = (tensor(g, sh, dt) for sh in (act(Ci, H, W), act(Ci, H, W), act(Co, Ho, Wo), act(Co, Ho, Wo)))
    w, dw = tensor(g, wsh, dt), tensor(g, wsh, dt)
    b, db = (tensor(g, (Co,), dt), tensor(g, (Co,), dt)) if bias else (None, None)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, Ci, H, W, Co, k, k, Ho, Wo, pad=(p, p, p, p), stride=(s, s), hwc=hwc, bias=b, dbias=db)
    chw = (lambda t: t.double().permute(0, 3, 1, 2)) if hwc else (lambda t: t.double())
    cols = F.unfold(chw(x), k, padding=p, stride=s)  # [ns][Ci k k][P]
    Wm, D = chw(w).reshape(Co, -1), chw(dy).reshape(ns, Co, -1)
    ref_y = (Wm @ cols).view(ns, Co, Ho, Wo) + (b.double().view(1, Co, 1, 1) if bias else 0)
    ref_dw = (D.permute(1, 0, 2).reshape(Co, -1) @ cols.permute(0, 2, 1).reshape(-1, Ci * k * k)).view(Co, Ci, k, k)
    ref_dx = F.fold(Wm.t() @ D, (H, W), k, padding=p, stride=s)
    gpu.ptl_set_gemm_path(7)
    try:
        for step, (tile, copies) in zip(("fw", "wg", "ig", "bw"), plans):
            for t in (y, dw, dx) + ((db,) if bias else ()):
                t.fill_(7)
            pkg.call("ptl_conv2d_%s_%s_batched" % (dt, step), a, ns)
            assert gpu.ptl_sync() == 0
            assert (gpu.ptl_last_gemm_tile(), gpu.ptl_last_conv_resident()) == (tile, 4 * copies), step
            if step == "fw":
                assert rel(chw(y), ref_y) <= TOL[dt]
            if step in ("wg", "bw"):
                assert rel(chw(dw), ref_dw) <= TOL[dt], step
                if bias:
                    assert rel(db, D.sum((0, 2))) <= TOL[dt], step
            if step in ("ig", "bw"):
                assert rel(chw(dx), ref_dx) <= TOL[dt], step
    finally:
        gpu.ptl_set_gemm_path(0)


T32 = 32032


@pytest.mark.parametrize("dt,N,M_,K,trans,tile", [("fp32", 1001, 1003, 777, 0, M), ("fp32", 1001, 1003, 777, 1, M), ("fp32", 999, 1001, 1003, 0, L),
                                                  ("fp32", 999, 1001, 1003, 1, L), ("fp16", 1001, 1003, 777, 0, M), ("fp16", 2049, 1030, 515, 0, L),
                                                  ("fp16", 2049, 1030, 515, 1, L), ("fp16", 700, 515, 900, 1, T32)])
def test_plain_products(pkg, gpu, dt, N, M_, K, trans, tile):
    g = torch.Generator(device=DEV).manual_seed(N)
    A, B, C = tensor(g, (N, K), dt), tensor(g, (M_, K) if trans else (K, M_), dt), tensor(g, (N, M_), dt)
    assert getattr(gpu, "ptl_mm_" + dt)(A.data_ptr(), B.data_ptr(), C.data_ptr(), N, M_, K, trans) == 0, gpu.ptl_last_error().decode()
    assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_tile() == tile
    assert rel(C, A.double() @ (B.double().t() if trans else B.double())) <= TOL[dt]


@pytest.mark.parametrize("dt,ns,n_in,n_out,tile", [("fp32", 391, 785, 333, T32), ("fp32", 300, 2001, 1003, M), ("fp32", 1000, 999, 1501, L),
                                                   ("fp16", 391, 785, 333, M), ("fp16", 2049, 700, 300, L)])
@pytest.mark.parametrize("bias", [0, 1])
def test_gradients_of_dense_layers(pkg, gpu, dt, ns, n_in, n_out, tile, bias):
    g = torch.Generator(device=DEV).manual_seed(ns)
    x, dx, w, dw, y, dy = (tensor(g, s, dt) for s in ((ns, n_in),) * 2 + ((n_out, n_in),) * 2 + ((ns, n_out),) * 2)
    b, db = (tensor(g, (n_out,), dt), tensor(g, (n_out,), dt)) if bias else (None, None)
    a, keep = hp.linear_args(pkg, x, dx, w, dw, y, dy, n_in, n_out, b, db)
    pkg.call("ptl_linear_%s_bw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_tile() == tile
    X, W, D = x.double(), w.double(), dy.double()
    assert rel(dw, D.t() @ X) <= TOL[dt] and rel(dx, D @ W) <= TOL[dt]
    if bias:
        assert rel(db, D.sum(0)) <= TOL[dt]
