"""Bias gradients are sums over all samples and positions: on every route no further from 64 bits than a tree of additions
by 256 threads, and infinities stay infinities."""
import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def tree_of_256(v):
    """Sum over the first axis in float32: 256 threads add every 256th value, then halves are added to halves."""
    n = v.shape[0]
    s = torch.zeros((256,) + v.shape[1:], dtype=torch.float32, device=v.device)
    for i in range(0, n, 256):
        part = v[i:i + 256]
        s[:part.shape[0]] += part
    while s.shape[0] > 1:
        s = s[:s.shape[0] // 2] + s[s.shape[0] // 2:]
    return s[0]


def check(db, values):
    """values: [positions][channels].  The bound is the tree's own error on these values, and at least what rounding the
    result once (2^-24 at most, half of that in the mean) and a handful of partial sums gives."""
    ref = values.double().sum(0)
    err = float((db.double() - ref).norm() / ref.norm())
    tree = float((tree_of_256(values).double() - ref).norm() / ref.norm())
    print("error %.2e, a tree of 256 %.2e" % (err, tree))
    assert err <= max(tree, 0.75 * 2.0 ** -24)


def run_dense(pkg, gpu, ns, n_in, n_out, dy, step):
    g = torch.Generator(device=DEV).manual_seed(ns)
    x, w = (torch.rand(s, generator=g, device=DEV).to(dy.dtype) for s in ((ns, n_in), (n_out, n_in)))
    y, dx, dw, b, db = (torch.zeros(s, device=DEV, dtype=dy.dtype) for s in ((ns, n_out), (ns, n_in), (n_out, n_in), (n_out,), (n_out,)))
    a, keep = hp.linear_args(pkg, x, dx, w, dw, y, dy, n_in, n_out, b, db)
    pkg.call("ptl_linear_%s_%s_batched" % ("fp32" if dy.dtype == torch.float32 else "fp16", step), a, ns)
    assert gpu.ptl_sync() == 0
    return db


# one launch with tiles of 32, 64 and 128 and with a split contraction; the kernels that sum rows, with and without shares
DENSE = [(391, 785, 333, "bw"), (512, 64, 1024, "bw"), (512, 33, 70, "bw"), (8192, 64, 10, "bw"), (1000, 999, 1501, "bw"),
         (2048, 1024, 1024, "bw"), (512, 64, 100, "wg"), (4096, 8, 32768, "wg"), (20000, 16, 24, "wg"), (7, 5, 9, "bw")]


@pytest.mark.parametrize("ns,n_in,n_out,step", DENSE)
def test_dense_layers(pkg, gpu, ns, n_in, n_out, step):
    dy = torch.rand((ns, n_out), generator=torch.Generator(device=DEV).manual_seed(n_in), device=DEV)
    check(run_dense(pkg, gpu, ns, n_in, n_out, dy, step), dy)


# samples, Ci, Co, H, W, kernel, stride, channel-minor, path: whole images as runs of k, all pixels as one, tiles of all sizes,
# channel-minor copies of the tensors; the kernel that sums planes (behind the small layers' kernel)
CONV = [(33, 24, 45, 57, 57, 5, 2, 0, 7), (8, 16, 24, 32, 32, 3, 1, 0, 7), (64, 40, 96, 13, 13, 3, 1, 0, 7), (16, 24, 40, 31, 30, 3, 1, 1, 7),
        (128, 128, 128, 14, 14, 3, 1, 1, 7), (64, 96, 256, 14, 14, 3, 1, 0, 7), (64, 16, 16, 32, 32, 3, 1, 0, 0), (3, 8, 16, 9, 9, 3, 1, 0, 1),
        (200, 8, 24, 17, 17, 3, 1, 1, 1)]


@pytest.mark.parametrize("ns,Ci,Co,H,W,k,s,hwc,path", CONV)
def test_convolutions(pkg, gpu, ns, Ci, Co, H, W, k, s, hwc, path):
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci)
    act = (lambda c, h, w: (ns, h, w, c)) if hwc else (lambda c, h, w: (ns, c, h, w))
    x, dy = torch.rand(act(Ci, H, W), generator=g, device=DEV), torch.rand(act(Co, Ho, Wo), generator=g, device=DEV)
    wsh = (Co, k, k, Ci) if hwc else (Co, Ci, k, k)
    w, dw, y, dx, b, db = (torch.zeros(sh, device=DEV) for sh in (wsh, wsh, dy.shape, x.shape, (Co,), (Co,)))
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, Ci, H, W, Co, k, k, Ho, Wo, pad=(p, p, p, p), stride=(s, s), hwc=hwc, bias=b, dbias=db)
    gpu.ptl_set_gemm_path(path)
    try:
        pkg.call("ptl_conv2d_fp32_wg_batched", a, ns)
        assert gpu.ptl_sync() == 0
    finally:
        gpu.ptl_set_gemm_path(0)
    check(db, dy.reshape(-1, Co) if hwc else dy.permute(0, 2, 3, 1).reshape(-1, Co))


@pytest.mark.parametrize("ns,n_in,n_out,step", [(391, 785, 333, "bw"), (8192, 64, 10, "bw"), (512, 64, 100, "wg"), (20000, 16, 24, "wg")])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_infinities(pkg, gpu, dt, ns, n_in, n_out, step):
    dy = torch.rand((ns, n_out), generator=torch.Generator(device=DEV).manual_seed(n_in), device=DEV).to(dt)
    inf = float("inf")
    dy[ns // 3, 1], dy[ns - 1, 2], dy[0, 3], dy[ns // 2, 3], dy[5, 4] = inf, -inf, inf, -inf, float("nan")
    db = run_dense(pkg, gpu, ns, n_in, n_out, dy, step)
    assert float(db[1]) == inf and float(db[2]) == -inf and bool(db[3:5].isnan().all())
    assert bool(db[0].isfinite()) and bool(db[5:].isfinite().all())


# both gradients in one launch, by whole images and by pixels, on copies, channel-minor in pieces, of one tap, tiles of 32 to 128
BOTH = [(57, 35, 40, 15, 15, 5, 1, 0, 0), (72, 8, 40, 23, 23, 3, 2, 0, 0), (49, 244, 33, 10, 10, 1, 1, 0, 0), (9, 20, 45, 5, 5, 3, 1, 0, 0),
        (20, 39, 72, 19, 19, 1, 1, 1, 0), (30, 24, 40, 21, 20, 3, 1, 1, 0), (13, 64, 150, 16, 16, 3, 1, 0, 9), (64, 96, 256, 14, 14, 3, 1, 0, 7),
        (33, 24, 45, 57, 57, 5, 2, 0, 0), (40, 64, 256, 30, 30, 1, 1, 0, 0)]


@pytest.mark.parametrize("ns,Ci,Co,H,W,k,s,hwc,path", BOTH)
def test_backward_calls_of_convolutions_round_once(pkg, gpu, ns, Ci, Co, H, W, k, s, hwc, path):
    """Values of both signs, so that the sums are small beside their terms."""
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    g = torch.Generator(device=DEV).manual_seed(Ci)
    act = (lambda c, h, w: (ns, h, w, c)) if hwc else (lambda c, h, w: (ns, c, h, w))
    x, dy = (torch.rand(sh, generator=g, device=DEV) * 2 - 1 for sh in (act(Ci, H, W), act(Co, Ho, Wo)))
    wsh = (Co, k, k, Ci) if hwc else (Co, Ci, k, k)
    w, dw, y, dx, b, db = (torch.zeros(sh, device=DEV) for sh in (wsh, wsh, dy.shape, x.shape, (Co,), (Co,)))
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, y, dy, Ci, H, W, Co, k, k, Ho, Wo, pad=(p, p, p, p), stride=(s, s), hwc=hwc, bias=b, dbias=db)
    gpu.ptl_set_gemm_path(path)
    try:
        pkg.call("ptl_conv2d_fp32_bw_batched", a, ns)
        assert gpu.ptl_sync() == 0
    finally:
        gpu.ptl_set_gemm_path(0)
    ref = (dy.reshape(-1, Co) if hwc else dy.permute(0, 2, 3, 1).reshape(-1, Co)).double().sum(0)
    # the rounding of a result is 2^-24 of it at most, 0.42 of that in the root mean square over all mantissas
    assert float((db.double() - ref).norm() / ref.norm()) <= 0.6 * 2.0 ** -24


@pytest.mark.parametrize("ns,n_in,n_out", [(2, 1, 77), (3, 600, 130), (4, 86, 259), (5, 4100, 65), (7, 177, 646), (8, 144, 1001)])
def test_few_samples_round_once(pkg, gpu, ns, n_in, n_out):
    dy = torch.rand((ns, n_out), generator=torch.Generator(device=DEV).manual_seed(n_in), device=DEV) * 2 - 1
    db = run_dense(pkg, gpu, ns, n_in, n_out, dy, "bw")
    assert gpu.ptl_last_gemm_form() == 3
    assert torch.equal(db, dy.double().sum(0).float())
