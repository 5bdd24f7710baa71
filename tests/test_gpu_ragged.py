"""Products whose sizes are no whole slabs or vectors and whose tensors start anywhere: the kernel for any size and
alignment (plain products, dense layers with biases in one launch, pointwise layers over planes that are no whole
vectors), at the edges of its tiles and pieces, against float64."""
import ctypes

import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {"fp32": 2e-6, "fp16": 1e-3}


def tensor(g, shape, dt, shift=0):
    """Uniform values at `shift` elements into a buffer whose other elements are NaN: nothing outside may be used."""
    tdt = torch.float32 if dt == "fp32" else torch.float16
    n = 1
    for s in shape:
        n *= s
    buf = torch.full((n + shift + 64,), float("nan"), dtype=tdt, device=DEV)
    t = buf[shift:shift + n].view(shape)
    t.copy_(torch.rand(shape, generator=g, device=DEV) * 2 - 1)
    return t


def rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("trans", [0, 1])
# one element over and under a tile, a slab, a piece; k shorter than a slab; a k split; rows shorter than a piece
@pytest.mark.parametrize("N,M,K,shift", [(33, 65, 65, 0), (31, 63, 127, 1), (129, 127, 33, 3), (300, 201, 2051, 1), (64, 9, 70, 0),
                                         (8, 8, 8, 1), (9, 1030, 9, 5), (5, 3, 700, 1), (700, 3, 5, 1),
                                         # one row: columns summed in shares of the rows (the last of 2, of 8, of 32; none)
                                         (1, 2049, 8193, 1), (1, 257, 4097, 0), (1, 67, 16411, 3), (1, 10, 8195, 1), (1, 3, 4096, 0)])
def test_plain_products(pkg, gpu, dt, trans, N, M, K, shift):
    g = torch.Generator(device=DEV).manual_seed(N * 7 + M)
    A, B = tensor(g, (N, K), dt, shift), tensor(g, (M, K) if trans else (K, M), dt, shift)
    Cm = tensor(g, (N, M), dt, shift)
    f = getattr(gpu, "ptl_mm_" + dt)
    assert f(A.data_ptr(), B.data_ptr(), Cm.data_ptr(), N, M, K, trans) == 0, gpu.ptl_last_error().decode()
    assert gpu.ptl_sync() == 0
    assert rel(Cm, A.double() @ (B.double().t() if trans else B.double())) <= TOL[dt]


def test_outer_product_of_more_pieces_than_31_bits_count(pkg, gpu):
    """A column times a row, 65 540 x 1 048 584 in fp16: 137 GB, 2^31 units of four rows x one piece and some more."""
    N, M = 65540, (1 << 20) + 8
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 160e9:
        pytest.skip("less than 160 GB of memory free")
    a = (torch.arange(N, device=DEV) % 31).to(torch.float16)  # (products are whole numbers below 2^11: exact)
    b = (torch.arange(M, device=DEV) % 61).to(torch.float16)
    C = torch.full((N, M), -1, dtype=torch.float16, device=DEV)
    assert gpu.ptl_mm_fp16(a.data_ptr(), b.data_ptr(), C.data_ptr(), N, M, 1, 0) == 0, gpu.ptl_last_error().decode()
    assert gpu.ptl_sync() == 0
    for r in range(0, N, 4096):
        assert bool((C[r:r + 4096] == a[r:r + 4096].view(-1, 1) * b).all()), r
    del C
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("ns,n_in,n_out,shift", [(1, 33, 9, 1), (1, 5, 3, 0), (1, 4101, 5, 3), (2, 64, 10, 0), (33, 127, 65, 1),
                                                (391, 785, 333, 0), (5000, 40, 12, 0), (3, 6, 5, 0), (130, 513, 256, 0),
                                                (1, 71, 16387, 1), (1, 1031, 4099, 0), (1, 6, 9001, 1)])
@pytest.mark.parametrize("bias", [0, 1])
def test_dense_layers(pkg, gpu, dt, ns, n_in, n_out, shift, bias):
    g = torch.Generator(device=DEV).manual_seed(ns + n_in)
    x, w, dy = tensor(g, (ns, n_in), dt, shift), tensor(g, (n_out, n_in), dt, shift), tensor(g, (ns, n_out), dt, shift)
    y, dx, dw = tensor(g, (ns, n_out), dt, shift), tensor(g, (ns, n_in), dt, shift), tensor(g, (n_out, n_in), dt, shift)
    b, db = (tensor(g, (n_out,), dt, shift), tensor(g, (n_out,), dt, shift)) if bias else (None, None)
    a, keep = hp.linear_args(pkg, x, dx, w, dw, y, dy, n_in, n_out, b, db)
    pkg.call("ptl_linear_%s_fw_batched" % dt, a, ns)
    pkg.call("ptl_linear_%s_bw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    X, W, D = x.double(), w.double(), dy.double()
    assert rel(y, X @ W.t() + (b.double() if bias else 0)) <= TOL[dt]
    assert rel(dw, D.t() @ X) <= TOL[dt]
    assert rel(dx, D @ W) <= TOL[dt]
    if bias:
        assert rel(db, D.sum(0)) <= TOL[dt]


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("ns,Ci,Co,H,W", [(3, 9, 17, 5, 7), (2, 33, 65, 13, 13), (5, 64, 10, 7, 9), (130, 8, 12, 3, 3)])
@pytest.mark.parametrize("hwc", [0, 1])
def test_pointwise_layers(pkg, gpu, dt, ns, Ci, Co, H, W, hwc):
    g = torch.Generator(device=DEV).manual_seed(Ci * Co)
    sh = (lambda c: (ns, H, W, c)) if hwc else (lambda c: (ns, c, H, W))
    x, dy, w = tensor(g, sh(Ci), dt), tensor(g, sh(Co), dt), tensor(g, (Ci, Co) if hwc and dt == "fp32" else (Co, Ci), dt)
    y, dx, dw = tensor(g, sh(Co), dt), tensor(g, sh(Ci), dt), tensor(g, tuple(w.shape), dt)
    a, keep = hp.pw_args(pkg, x, dx, w, dw, y, dy, Ci, Co, H, W, hwc)
    for step in ("fw", "wg", "ig"):
        pkg.call("ptl_conv_pw_%s_%s_batched" % (dt, step), a, ns)
    assert gpu.ptl_sync() == 0
    flat = (lambda t, c: t.double().reshape(-1, c)) if hwc else (lambda t, c: t.double().permute(0, 2, 3, 1).reshape(-1, c))
    X, D, Wm = flat(x, Ci), flat(dy, Co), w.double() if hwc and dt == "fp32" else w.double().t()  # Wm: [Ci][Co]
    gw = dw.double() if hwc and dt == "fp32" else dw.double().t()
    assert rel(flat(y, Co), X @ Wm) <= TOL[dt]
    assert rel(flat(dx, Ci), D @ Wm.t()) <= TOL[dt]
    assert rel(gw, X.t() @ D) <= TOL[dt]


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("ns,C,H,W,hwc", [(1, 3, 5, 5, 0), (2, 5, 300, 300, 0), (70, 6, 13, 7, 0), (9, 65, 20, 21, 1), (3, 130, 9, 9, 1)])
def test_bias_and_bias_gradient_of_a_convolution(pkg, gpu, dt, ns, C, H, W, hwc):
    """1x1 layer with an identity filter: y = x + bias; the bias gradient is a sum over all positions."""
    g = torch.Generator(device=DEV).manual_seed(C + H)
    sh = (ns, H, W, C) if hwc else (ns, C, H, W)
    x, dy, y, dx = (tensor(g, sh, dt) for _ in range(4))
    w, dw, b, db = torch.eye(C, device=DEV).to(x.dtype), tensor(g, (C, C), dt), tensor(g, (C,), dt), tensor(g, (C,), dt)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, C, H, W, C, 1, 1, H, W, hwc=hwc, bias=b, dbias=db)
    pkg.call("ptl_conv2d_%s_fw_batched" % dt, a, ns)
    pkg.call("ptl_conv2d_%s_bw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    bb = b.double() if hwc else b.double().view(1, C, 1, 1)
    assert rel(y, x.double() + bb) <= TOL[dt]
    assert rel(db, dy.double().sum((0, 1, 2) if hwc else (0, 2, 3))) <= 10 * TOL[dt]
