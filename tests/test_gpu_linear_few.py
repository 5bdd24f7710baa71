"""Dense layers on a few samples: weights read once for all of them, sums of rows and of columns in 16-byte pieces."""
import pytest
import torch

from test_gpu_patch_rows import DEV, shifted

pytestmark = pytest.mark.gpu
TDT = {"fp32": torch.float32, "fp16": torch.float16}


def run(pkg, gpu, dt, ns, n_in, n_out, bias, shift, spoil=None, takes=None):
    g = torch.Generator(device=DEV).manual_seed(n_in * 31 + n_out)
    r = lambda *s: shifted((torch.rand(*s, generator=g, device=DEV) - 0.5).to(TDT[dt]), shift)[0]
    x, w, b, dy = r(ns, n_in), r(n_out, n_in), r(n_out), r(ns, n_out)
    if spoil:
        w[spoil], x[:, 0] = float("inf"), 1.0
    guard = {k: shifted(torch.zeros(*s, device=DEV, dtype=TDT[dt]), shift) for k, s in
             (("y", (ns, n_out)), ("dx", (ns, n_in)), ("dw", (n_out, n_in)), ("db", (n_out,)))}
    y, dx, dw, db = (guard[k][0] for k in ("y", "dx", "dw", "db"))
    a = pkg.LinearArgs()
    keep = [pkg.blob(x, dx, 1, 1, 1, n_in), pkg.blob(w, dw, 1, 1, 1, n_in * n_out), pkg.blob(b, db, 1, 1, 1, n_out), pkg.blob(y, dy, 1, 1, 1, n_out)]
    a.input, a.coeff, a.bias, a.output = [pkg.structs.C.pointer(k) for k in keep]
    a.use_biases = bias
    for k, q in zip(keep, (n_in, n_in * n_out, n_out, n_out)):
        assert k.dim == q
    pkg.call("ptl_linear_%s_fw_batched" % dt, a, ns)
    forms = [gpu.ptl_last_gemm_form()]
    pkg.call("ptl_linear_%s_bw_batched" % dt, a, ns)
    assert gpu.ptl_sync() == 0
    forms.append(gpu.ptl_last_gemm_form())
    few_bw = ns <= 8 and (dt == "fp32" or ns <= 4 or ((n_in >= 1024 or n_out >= 1536) and n_in <= 128 * n_out))
    assert [f == 3 for f in forms] == list(takes or (ns <= 8 or n_out <= 1280, few_bw))
    for t, buf in guard.values():
        assert bool((buf[:shift] == 5).all()) and bool((buf[shift + t.numel():] == 5).all())
    X, W, B, D = (t.double() for t in (x, w, b, dy))
    ref = {"y": X @ W.t() + (B if bias else 0), "dx": D @ W, "dw": D.t() @ X, "db": D.sum(0) if bias else torch.zeros_like(B)}
    size = {"y": X.abs() @ W.abs().t() + B.abs(), "dx": D.abs() @ W.abs(), "dw": D.abs().t() @ X.abs(), "db": D.abs().sum(0)}
    return {"y": y, "dx": dx, "dw": dw, "db": db}, ref, size


def check(dt, got, ref, size, n_in, n_out):
    for k, v in got.items():
        # a chain of roundings: the terms of a lane's sum (a 64th of the contraction), of a wave's and of the waves
        chain = {"y": n_in / 64, "dx": n_out / 64}.get(k, 0) + 40
        tol = chain * 2.0 ** -24 * size[k] + (2.0 ** -11 * ref[k].abs() + 2.0 ** -25 if dt == "fp16" else 0)
        assert bool(((v.double() - ref[k]).abs() <= tol).all()), k


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("ns", [2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n_in,n_out,bias,shift", [(1, 5, 1, 0), (3, 9, 0, 1), (7, 1, 1, 1), (8, 8, 1, 0), (9, 65, 0, 1), (255, 63, 1, 3), (257, 64, 0, 0),
                                                   (513, 521, 1, 1), (1025, 130, 0, 0), (2049, 7, 1, 1), (300, 2050, 1, 0), (70, 1100, 0, 1),
                                                   (1031, 1033, 1, 1)])
def test_few_samples(pkg, gpu, dt, ns, n_in, n_out, bias, shift):
    check(dt, *run(pkg, gpu, dt, ns, n_in, n_out, bias, shift), n_in, n_out)


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("ns", [2, 4, 7])
def test_rows_shared_out(pkg, gpu, dt, ns):
    """1536 rows and more: shares of the column sums that a second launch adds."""
    n_in, n_out = 520, 1541
    check(dt, *run(pkg, gpu, dt, ns, n_in, n_out, 1, 1), n_in, n_out)


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("n_in,n_out", [(70, 77), (600, 530)])
def test_infinite_weights_stay_in_their_row_and_column(pkg, gpu, dt, n_in, n_out):
    """What is read in place of rows and pieces beyond the end does not count: the last row and column hold infinities."""
    ns = 3
    got, ref, size = run(pkg, gpu, dt, ns, n_in, n_out, 0, 1, spoil=(n_out - 1, n_in - 1))
    for k in ("y", "dx"):
        assert torch.equal(got[k].isfinite(), ref[k].isfinite()) and torch.equal(got[k].isnan(), ref[k].isnan())
        fin = ref[k].isfinite()
        got[k], ref[k], size[k] = got[k][fin], ref[k][fin], size[k][fin]
    check(dt, got, ref, size, n_in, n_out)


@pytest.mark.parametrize("dt,ns,n_in,n_out,fw,bw", [
    ("fp32", 4, 4096, 4096, 1, 1), ("fp32", 3, 4352, 4096, 0, 1),      # 70 MB of weights
    ("fp16", 8, 2928, 4096, 1, 1), ("fp16", 5, 2936, 4096, 0, 1),      # 24 MB
    ("fp32", 8, 16384, 64, 1, 1), ("fp32", 8, 16388, 64, 0, 1),        # long rows
    ("fp32", 16, 1024, 1280, 1, 0), ("fp32", 9, 1076, 1280, 0, 0),     # 5.5 MB
    ("fp16", 16, 4096, 64, 1, 0), ("fp16", 9, 4104, 64, 0, 0), ("fp32", 12, 3076, 64, 0, 0), ("fp16", 9, 512, 1281, 0, 0),
    ("fp32", 2, 255, 4096, 1, 1), ("fp32", 2, 255, 4097, 0, 1), ("fp32", 8, 256, 4097, 1, 1),  # many short rows
    ("fp16", 2, 2048, 8193, 1, 1), ("fp16", 2, 2040, 8193, 0, 1), ("fp16", 4, 2048, 8193, 0, 1),
    ("fp32", 4, 512, 16384, 1, 1), ("fp32", 4, 511, 16384, 0, 1), ("fp32", 4, 512, 16385, 0, 1), ("fp32", 5, 512, 8193, 0, 1),
    ("fp16", 8, 8192, 64, 1, 1), ("fp16", 8, 8200, 64, 1, 0), ("fp16", 8, 20, 10240, 0, 1), ("fp16", 8, 20, 10248, 0, 0)])
def test_lines_to_the_other_routes(pkg, gpu, dt, ns, n_in, n_out, fw, bw):
    check(dt, *run(pkg, gpu, dt, ns, n_in, n_out, 1, 0, takes=(fw, bw)), n_in, n_out)


def test_more_outputs_than_one_launch_of_row_sums_has_threads_for(pkg, gpu):
    """2^26 rows, a wave each: such a launch left the outputs as they were."""
    ns, n_out = 2, 2 ** 26 + 5
    x, w = torch.tensor([[2.0], [-3.0]], device=DEV).half(), (torch.arange(n_out, device=DEV) % 511).half()
    y = torch.zeros(ns, n_out, device=DEV).half()
    a = pkg.LinearArgs()
    keep = [pkg.blob(x, None, dim=1), pkg.blob(w, None, dim=n_out), pkg.blob(y, None, dim=n_out)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(k) for k in keep]
    pkg.call("ptl_linear_fp16_fw_batched", a, ns)
    assert gpu.ptl_sync() == 0
    assert torch.equal(y, x * w)
