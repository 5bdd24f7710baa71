"""fp32 dense layers on 128 x 128 tiles whose contraction is cut into fewer parts so that they run as bf16 pieces, and neighbours that
keep their parts: tile, form and results against float64."""
import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# samples, in, out, direction, form (1: bf16 pieces).  The last two: too few workgroups, hardly fewer clocks
@pytest.mark.parametrize("case", [(2048, 1000, 1001, "fw", 1), (2993, 734, 1095, "fw", 1), (507, 2297, 2112, "fw", 1), (4565, 2012, 256, "fw", 1),
                                  (511, 1023, 2047, "bw", 1), (448, 1643, 1280, "bw", 1), (511, 1023, 2047, "fw", 0), (3031, 1280, 415, "bw", 0)])
def test_parts(pkg, gpu, case):
    ns, n_in, n_out, step, form = case
    g = torch.Generator(device=DEV).manual_seed(ns)
    x, w, dy = (torch.rand(s, generator=g, device=DEV) * 2 - 1 for s in ((ns, n_in), (n_out, n_in), (ns, n_out)))
    y, dx, dw = torch.full_like(dy, 7), torch.full_like(x, 7), torch.full_like(w, 7)
    a, keep = hp.linear_args(pkg, x, dx, w, dw, y, dy, n_in, n_out)
    X, W, D = x.double(), w.double(), dy.double()
    pkg.call("ptl_linear_fp32_%s_batched" % step, a, ns)
    assert gpu.ptl_sync() == 0
    assert (gpu.ptl_last_gemm_tile(), gpu.ptl_last_gemm_form()) == (128128, form)
    for got, want in ((y, X @ W.T),) if step == "fw" else ((dw, D.T @ X), (dx, D @ W)):
        # sums of sums of 32 terms, each addition rounded by 2^-24 at most: 1.2e-7 in the mean, as in the tests of fp32 sums
        assert float((got.double() - want).norm() / want.norm()) <= 4e-7


@pytest.mark.parametrize("what", ["infinity", "nan", "huge", "tiny"])
@pytest.mark.parametrize("case", [(2993, 734, 1095, "fw"), (511, 1023, 2047, "bw")])
def test_values_outside_the_range_of_the_pieces(pkg, gpu, case, what):
    """One such value in each operand; a tile without one keeps the bits that it has without them."""
    ns, n_in, n_out, step = case
    g = torch.Generator(device=DEV).manual_seed(ns)
    x, w, dy = (torch.rand(s, generator=g, device=DEV) * 2 - 1 for s in ((ns, n_in), (n_out, n_in), (ns, n_out)))
    outs = lambda: (torch.full_like(dy, 7), torch.full_like(x, 7), torch.full_like(w, 7))

    def run():
        y, dx, dw = outs()
        a, keep = hp.linear_args(pkg, x, dx, w, dw, y, dy, n_in, n_out)
        pkg.call("ptl_linear_fp32_%s_batched" % step, a, ns)
        assert gpu.ptl_sync() == 0 and (gpu.ptl_last_gemm_tile(), gpu.ptl_last_gemm_form()) == (128128, 1)
        return (y,) if step == "fw" else (dw, dx)

    plain = run()
    first, second = (x, w) if step == "fw" else (dy, x)
    if what == "tiny":  # (the third piece of 1e-35 would lie below the smallest bf16)
        first.mul_(1e-35)
    else:  # (huge: rounds up to infinity as a bf16)
        value = {"infinity": float("inf"), "nan": float("nan"), "huge": 3.4e38}[what]
        first[300, 400], second[200, 500] = value, -value
        if what == "huge":
            second.mul_(0.25)
    X, W, D = x.double(), w.double(), dy.double()
    for got, kept, ref in zip(run(), plain, (X @ W.T,) if step == "fw" else (D.T @ X, D @ W)):
        if what in ("infinity", "nan"):  # (the values reach rows 300 and 400 and columns 200 and 500)
            assert torch.equal(got[:128, :128], kept[:128, :128])
        got = got.double()
        ref = torch.where(ref.abs() > torch.finfo(torch.float32).max, ref * float("inf"), ref)
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])
        fin = ref.isfinite()
        size = ref[fin].abs().max() if what == "huge" else (ref[fin] ** 2).mean().sqrt()
        # up to 2047 products, 64 slabs: sqrt(64 / 3) roundings of 2^-25 and of 2^-24 in eight, six times that for the largest of 3 million
        assert float((got[fin] - ref[fin]).abs().max()) <= 4e-6 * float(size)
