"""Shallow products: the column tiles of a panel shared out over its workgroups, from fewer than the XCDs to many."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TDT = {"fp32": torch.float32, "fp16": torch.float16}


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
# tiles of 64 columns by panels of 64 or 128 rows: 1, 2, 7, 8, 9, 10, 17 and 87 tiles
@pytest.mark.parametrize("n_in,ns", [(40, 33000), (65, 20000), (448, 5000), (512, 5000), (513, 5001), (577, 8733), (1081, 4097), (5519, 1300)])
def test_input_gradient(pkg, gpu, dt, n_in, ns):
    n_out = 33
    g = torch.Generator(device=DEV).manual_seed(n_in)
    r = lambda *s: (torch.rand(*s, generator=g, device=DEV) - 0.5).to(TDT[dt])
    w, dy, x = r(n_out, n_in), r(ns, n_out), r(ns, n_in)
    buf = torch.full((ns * n_in + 64,), 5.0, device=DEV, dtype=TDT[dt])
    dx = buf[:-64]
    a = pkg.LinearArgs()
    keep = [pkg.blob(x, dx, dim=n_in), pkg.blob(w, None, dim=n_in * n_out), pkg.blob(None, dy, dim=n_out)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(k) for k in keep]
    pkg.call("ptl_linear_%s_ig_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    assert bool((buf[-64:] == 5).all())
    W, D = w.double(), dy.double()
    ref, size = D @ W, D.abs() @ W.abs()
    # one rounding a term, one at the end
    tol = n_out * 2.0 ** -24 * size + (2.0 ** -11 * ref.abs() + 2.0 ** -25 if dt == "fp16" else 0)
    assert bool(((dx.view(ns, n_in).double() - ref).abs() <= tol).all())
