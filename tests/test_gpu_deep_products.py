"""Products of few tiles with the contraction shared out over the waves of a tile, at the edges of pieces, steps, trips and
tiles, from the C API's forward pass of dense layers."""
import math

import pytest
import torch

from test_gpu_patch_rows import DEV, shifted

pytestmark = pytest.mark.gpu
TDT = {"fp32": torch.float32, "fp16": torch.float16}


def forward(pkg, gpu, dt, x, w, b, shift):
    (ns, n_in), n_out = x.shape, w.shape[0]
    y, buf = shifted(torch.zeros(ns, n_out, device=DEV, dtype=TDT[dt]), shift)
    a = pkg.LinearArgs()
    keep = [pkg.blob(x, None, dim=n_in), pkg.blob(w, None, dim=n_in * n_out), pkg.blob(b, None, dim=n_out), pkg.blob(y, None, dim=n_out)]
    a.input, a.coeff, a.bias, a.output = [pkg.structs.C.pointer(k) for k in keep]
    a.use_biases = int(b is not None)
    pkg.call("ptl_linear_%s_fw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    assert bool((buf[:shift] == 5).all()) and bool((buf[shift + y.numel():] == 5).all())
    return y


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("ns,n_out", [(17, 2), (31, 33), (32, 32), (33, 31), (65, 97), (300, 20)])
@pytest.mark.parametrize("n_in", [4, 5, 8, 10, 16, 18, 30, 62, 64, 66, 254, 258, 510, 514, 769, 1022, 1024])
def test_edges(pkg, gpu, dt, ns, n_out, n_in):
    shift = 2 if n_in % 3 else 0
    g = torch.Generator(device=DEV).manual_seed(n_in * 1000 + ns)
    r = lambda *s: shifted((torch.rand(*s, generator=g, device=DEV) - 0.5).to(TDT[dt]), shift)[0]
    x, w, b = r(ns, n_in), r(n_out, n_in), (r(n_out) if ns & 1 else None)
    y = forward(pkg, gpu, dt, x, w, b, shift)
    takes = 4 <= n_in <= 900 if dt == "fp32" else n_in >= 8 and n_in % 2 == 0
    assert (gpu.ptl_last_gemm_form() == 2) == takes
    X, W, B = x.double(), w.double(), 0 if b is None else b.double()
    ref, size = X @ W.t() + B, X.abs() @ W.abs().t() + abs(B)
    # a wave's chain of n_in / 8 additions at most, the sum of eight waves and the bias
    tol = (n_in / 8 + 10) * 2.0 ** -24 * size + (2.0 ** -11 * ref.abs() + 2.0 ** -25 if dt == "fp16" else 0)
    assert bool(((y.double() - ref).abs() <= tol).all())


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("n_in", [18, 102, 246, 390])
def test_what_is_cut_away_does_not_count(pkg, gpu, dt, n_in):
    """An infinity as the last element of a row is read again in pieces that are shifted out."""
    g = torch.Generator(device=DEV).manual_seed(n_in)
    x, w = ((torch.rand(s, n_in, generator=g, device=DEV) + 0.5).to(TDT[dt]) for s in (40, 50))
    x[7, n_in - 1], w[11, n_in - 1], x[39, 0] = float("inf"), -float("inf"), float("nan")
    y = forward(pkg, gpu, dt, x, w, None, 0)
    assert gpu.ptl_last_gemm_form() == 2
    ref = x.double() @ w.double().t()
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    fin = ref.isfinite()
    assert bool(((y.double() - ref).abs()[fin] <= (2.0 ** -10 if dt == "fp16" else 2e-5) * ref[fin]).all())


@pytest.mark.parametrize("ns,n_in,n_out", [(100, 65, 333), (100, 513, 128), (391, 785, 333), (391, 900, 200), (391, 901, 200)])
def test_sums_are_no_chains(pkg, gpu, ns, n_in, n_out):
    """fp32: a wave has four chains.  Roundings of at most u = 2^-24 leave u / sqrt(3) * sqrt(n / 2) after a chain of n additions of
    values of random sign; here a 32nd of the contraction, two more in a wave and the eight waves (beyond 900 slabs of 32)."""
    g = torch.Generator(device=DEV).manual_seed(n_in)
    x, w = (torch.rand(s, n_in, generator=g, device=DEV) * 2 - 1 for s in (ns, n_out))
    y = forward(pkg, gpu, "fp32", x, w, None, 0)
    assert gpu.ptl_last_gemm_form() == (2 if n_in <= 900 else 0)
    ref = x.double() @ w.double().t()
    bound = 2.0 ** -24 / math.sqrt(3) * math.sqrt((n_in / 32 + 10) / 2)
    assert float((y.double() - ref).norm() / ref.norm()) <= bound


@pytest.mark.parametrize("dt,n_in,n_out,takes", [
    ("fp32", 512, 864, 1), ("fp32", 496, 864, 0), ("fp32", 608, 864, 0), ("fp32", 800, 864, 0), ("fp32", 799, 864, 1), ("fp32", 801, 864, 0),
    ("fp32", 800, 512, 1), ("fp32", 20, 1376, 0), ("fp16", 64, 864, 1), ("fp16", 128, 864, 0), ("fp16", 130, 864, 1), ("fp16", 192, 864, 0),
    ("fp16", 192, 512, 1), ("fp16", 258, 864, 0)])
def test_lines_to_the_other_routes(pkg, gpu, dt, n_in, n_out, takes):
    """378 samples: twelve tiles in height, 192 to 516 of them on 256 compute units."""
    g = torch.Generator(device=DEV).manual_seed(n_in)
    x, w = ((torch.rand(s, n_in, generator=g, device=DEV) - 0.5).to(TDT[dt]) for s in (378, n_out))
    y = forward(pkg, gpu, dt, x, w, None, 0)
    assert (gpu.ptl_last_gemm_form() == 2) == takes
    ref = x.double() @ w.double().t()
    # fp32: as above, and one chain of additions on routes that look nothing up; fp16: roundings of the result, 2^-12 in the mean
    bound = 2.0 ** -24 / math.sqrt(3) * math.sqrt((n_in / 32 + 10 if takes else n_in) / 2)
    assert float((y.double() - ref).norm() / ref.norm()) <= (bound if dt == "fp32" else 2.5e-4)
