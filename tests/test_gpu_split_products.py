"""fp32 products formed from three bf16 pieces of each value: infinities and values above the pieces' range go through the fp32
instructions, small ones keep their bits, and the bf16 instructions' rounding (towards minus infinity) does not add up over long contractions."""
import pytest
import torch

import helpers as hp
from test_gpu_conv_any import rel, tensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def point_layer(pkg, ns, Ci, Co, P, g):
    x, dx, dy = tensor(g, (ns, Ci, 1, P), "fp32"), tensor(g, (ns, Ci, 1, P), "fp32"), tensor(g, (ns, Co, 1, P), "fp32")
    w, dw = tensor(g, (Co, Ci), "fp32"), tensor(g, (Co, Ci), "fp32")
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, dy, dy, Ci, 1, P, Co, 1, 1, 1, P, (0, 0, 0, 0), (1, 1), 0)
    return x, dx, dy, w, dw, a, keep


@pytest.mark.parametrize("what", ["infinity", "nan", "huge", "tiny"])
def test_values_outside_the_range_of_the_pieces(pkg, gpu, what):
    g = torch.Generator(device=DEV).manual_seed(3)
    ns, Ci, Co, P = 32, 270, 300, 333  # (contractions of 19 slabs and of 666: sixteen a workgroup or more take pieces)
    x, dx, dy, w, dw, a, keep = point_layer(pkg, ns, Ci, Co, P, g)
    if what == "tiny":  # (the third piece of 1e-35 would lie below the smallest bf16)
        x.mul_(1e-35)
        dy[:, 7].mul_(1e-2)
    else:  # (huge: rounds up to infinity as a bf16)
        x[2, 3, 0, 77] = {"infinity": float("inf"), "nan": float("nan"), "huge": 3.4e38}[what]
        dy[4, 9, 0, 5] = {"infinity": -float("inf"), "nan": float("nan"), "huge": -3.4e38}[what]
        if what == "huge":
            dy.mul_(0.25)
    pkg.call("ptl_conv2d_fp32_bw_batched", a, ns)
    assert gpu.ptl_sync() == 0 and (gpu.ptl_last_gemm_tile(), gpu.ptl_last_gemm_form()) == (64064, 1)
    X, D, W = x.double().reshape(ns, Ci, P), dy.double().reshape(ns, Co, P), w.double()
    ref_dw = sum(D[b] @ X[b].t().contiguous() for b in range(ns))
    ref_dx = torch.stack([W.t().contiguous() @ D[b] for b in range(ns)])
    for got, ref in ((dw, ref_dw), (dx.reshape(ns, Ci, P), ref_dx)):
        got = got.double()
        ref = torch.where(ref.abs() > torch.finfo(torch.float32).max, ref * float("inf"), ref)
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])
        fin = ref.isfinite()
        row = ref[fin].abs().max() if what == "huge" else (ref[fin] ** 2).mean().sqrt()
        # 10 700 products, 660 slabs: sqrt(660 / 3) roundings of 2^-25 and of 2^-24 in eight, five times that for the largest of 81 000
        assert float((got[fin] - ref[fin]).abs().max()) <= 4e-6 * float(row)
    if what == "tiny":  # row 7 by itself
        assert rel(dw[7], ref_dw[7]) <= 1e-6 and rel(dw[8], ref_dw[8]) <= 1e-6


def test_long_contractions_have_no_drift(pkg, gpu):
    """37 000 products a sum.  One rounding of 2^-25 towards minus infinity per instruction (six to 16 products) of sums of
    the size sqrt(32), added up, would be 3e-7 of a result; what is left of it when every other slab has the other sign is
    at most one slab's, 1e-8 or less."""
    g = torch.Generator(device=DEV).manual_seed(4)
    ns, Ci, Co, P = 64, 31, 300, 576
    x, dx, dy, w, dw, a, keep = point_layer(pkg, ns, Ci, Co, P, g)
    pkg.call("ptl_conv2d_fp32_bw_batched", a, ns)
    assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_form() == 1
    X, D = x.double().reshape(ns, Ci, P), dy.double().reshape(ns, Co, P)
    ref = sum(D[b] @ X[b].t().contiguous() for b in range(ns))
    err, rms = dw.double() - ref, float((ref ** 2).mean().sqrt())
    assert abs(float(err.mean())) <= 5e-8 * rms
    # random roundings: 8 slabs, then up to 50 sums of eight: sqrt((8 + 50) / 6) 2^-24 / sqrt(12) * 2, and a slab's own 7e-8
    assert rel(dw, ref) <= 2e-7


@pytest.mark.parametrize("hwc", [0, 1])
@pytest.mark.parametrize("ns", [39, 40])
def test_layers_on_both_sides_of_the_line_between_taps_and_patches(pkg, gpu, hwc, ns):
    """2.94 and 3.02 GFLOP: tap by tap, and as a product with patch matrices in bf16 pieces."""
    Ci = Co = 64
    H = W = 32
    g = torch.Generator(device=DEV).manual_seed(ns)
    act = (ns, H, W, Ci) if hwc else (ns, Ci, H, W)
    x, y, dy, w, dw = (torch.rand(s, generator=g, device=DEV) - 0.5 for s in (act, act, act, (Co, 3, 3, Ci) if hwc else (Co, Ci, 3, 3), (Co, 9 * Ci)))
    a, keep = hp.conv2d_args(pkg, x, dy, w, dw, y, dy, Ci, H, W, Co, 3, 3, H, W, pad=(1, 1, 1, 1), stride=(1, 1), hwc=hwc)
    pkg.call("ptl_conv2d_fp32_fw_batched", a, ns)
    assert gpu.ptl_sync() == 0
    assert (2e-9 * ns * Co * H * W * Ci * 9 >= 3) == (ns == 40)
    assert gpu.ptl_last_conv_direct() == (0 if ns == 40 else 1) and gpu.ptl_last_gemm_form() == (1 if ns == 40 else 0)
    chw = (lambda t: t.double().permute(0, 3, 1, 2)) if hwc else (lambda t: t.double())
    cols = torch.nn.functional.unfold(chw(x), 3, padding=1)
    ref = (chw(w).reshape(Co, -1) @ cols).view(ns, Co, H, W)
    # 576 products: sqrt(576 / 3) roundings of 2^-25 of a result's size
    assert rel(chw(y), ref) <= 4.2e-7


@pytest.mark.parametrize("ns,Ci,Co,k,stride", [(3, 24, 45, 5, 2), (9, 24, 45, 5, 2), (33, 24, 45, 5, 2), (18, 32, 38, 3, 1), (16, 4, 189, 3, 1)])
def test_weight_gradients_in_more_parts(pkg, gpu, ns, Ci, Co, k, stride):
    """Odd images, from contractions too short for bf16 pieces (up to nine samples) to ones in parts of some sixteen slabs."""
    H = W = 57
    Ho = (H + 2 * (k // 2) - k) // stride + 1
    g = torch.Generator(device=DEV).manual_seed(ns * Co)
    x, dy, w, dw = (torch.rand(s, generator=g, device=DEV) - 0.5 for s in ((ns, Ci, H, W), (ns, Co, Ho, Ho), (Co, Ci, k, k), (Co, Ci * k * k)))
    dx = torch.empty_like(x)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, dy, dy, Ci, H, W, Co, k, k, Ho, Ho, pad=(k // 2,) * 4, stride=(stride, stride), hwc=0)
    pkg.call("ptl_conv2d_fp32_bw_batched", a, ns)
    assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_form() == (1 if ns > 9 else 0)
    ref = torch.zeros(Co, Ci * k * k, dtype=torch.float64, device=DEV)
    for b in range(ns):
        cols = torch.nn.functional.unfold(x[b : b + 1].double(), k, padding=k // 2, stride=stride)[0]
        ref += dy[b].double().reshape(Co, -1) @ cols.t().contiguous()
    # as above, 2e-7, and up to 64 parts added up: sqrt(64 / 3) roundings of 2^-25
    assert rel(dw, ref) <= 3.4e-7


@pytest.mark.parametrize("size,other", [(-99, 60), (-112, 60), (-115, 60), (-120, 60), (-124, 60), (-130, 60), (-135, 60), (-149, 60), (-60, -60)])
@pytest.mark.parametrize("few", [0, 1])
def test_small_values_times_large_ones(pkg, gpu, size, other, few):
    """Values whose lower pieces, or that themselves, are below the smallest bf16 (2^-133), times ones of 2^60: results of 2^-40 to
    2^-85; and products that the smaller pieces leave below the smallest fp32 number.  few: one such value in a row, zeros beside it."""
    g = torch.Generator(device=DEV).manual_seed(5)
    ns, Ci, Co, P = 32, 270, 300, 333
    x, dx, dy, w, dw, a, keep = point_layer(pkg, ns, Ci, Co, P, g)
    dy.mul_(2.0 ** other)
    for t in (x, w):
        t.copy_(torch.where(t < 0, t - 1, t + 1) * 2.0 ** (size // 2) * 2.0 ** (size - size // 2))  # (1 to 2 times 2^size, with both signs)
    if few:
        one = x[3, :, 0, 50].clone()
        x.zero_()
        x[3, :, 0, 50] = one
    pkg.call("ptl_conv2d_fp32_bw_batched", a, ns)
    assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_form() == 1
    X, D, W = x.double().reshape(ns, Ci, P), dy.double().reshape(ns, Co, P), w.double()
    # sums as above, 2e-7 (one product: its rounding)
    assert rel(dw, sum(D[b] @ X[b].t().contiguous() for b in range(ns))) <= 2e-7
    assert rel(dx.reshape(ns, Ci, P), torch.stack([W.t().contiguous() @ D[b] for b in range(ns)])) <= 2e-7


def test_products_next_to_the_largest_number(pkg, gpu):
    """1.868e19 * 1.8205e19 = 3.4007e38 is finite, the product of the leading pieces is not."""
    g = torch.Generator(device=DEV).manual_seed(6)
    ns, Ci, Co, P = 32, 270, 300, 333
    x, dx, dy, w, dw, a, keep = point_layer(pkg, ns, Ci, Co, P, g)
    x.zero_()
    x[3, 7, 0, 50] = 1.868e19
    dy[3, 11, 0, 50] = 1.8205e19
    dy[3, 12, 0, 50] = -1.8205e19
    dy[3, 13, 0, 50] = 1.83e19
    pkg.call("ptl_conv2d_fp32_bw_batched", a, ns)
    assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_form() == 1
    ref = x[3, 7, 0, 50].double() * dy[3, :, 0, 50].double()
    assert float(dw[13, 7]) == float("inf") and float(ref[13]) > torch.finfo(torch.float32).max
    assert torch.equal(dw[:13, 7], ref[:13].float()) and float(ref[11]) == -float(ref[12])
