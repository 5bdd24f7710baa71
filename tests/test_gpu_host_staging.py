"""Host tensors: calls on them give the bits of the same calls on device tensors, whatever mix of small tensors (which
travel together through one pinned block) and large ones (a copy each) a call has."""
import numpy as np
import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (a byte-odd tensor; below, at and above the largest tensor of a block: 1 MiB; more than a block of 4 MiB in all)
@pytest.mark.parametrize("dt,n_in,n_out", [("fp16", 3, 5), ("fp32", 33, 65), ("fp32", 512, 512), ("fp32", 513, 512),
                                           ("fp16", 1000, 900)])
@pytest.mark.parametrize("skip", [(0, 0), (1, 0), (0, 1)])
def test_linear_on_host_arrays_matches_device(pkg, gpu, dt, n_in, n_out, skip):
    nd = hp.np_dtype(dt)
    x, w, dy = (hp.uniform(5 + i, s, dtype=nd) for i, s in enumerate(((n_in,), (n_out, n_in), (n_out,))))
    res = []
    for place in (lambda a: a.copy(), lambda a: torch.from_numpy(a).to(DEV)):
        t = [place(a) for a in (x, np.full(n_in, 3, nd), w, np.full((n_out, n_in), 3, nd), np.zeros(n_out, nd), dy)]
        a, keep = hp.linear_args(pkg, *t, n_in, n_out)
        a.skip_wg_grad, a.skip_in_grad = skip
        pkg.call("pulp_linear_%s_fw_cl" % dt, a)
        pkg.call("pulp_linear_%s_bw_cl" % dt, a)
        assert gpu.ptl_sync() == 0
        res.append([v if isinstance(v, np.ndarray) else v.cpu().numpy() for v in t])
    for h, d in zip(*res):
        assert np.array_equal(h, d)


def test_a_call_with_more_host_tensors_than_one_copy_kernel_takes(pkg, gpu):
    nd, opts, keep, ref = np.float32, [], [], []
    for i in range(45):  # 90 tensors, the last ones beyond the block
        n = 40000 if i > 12 else 7 + i
        w, dw = hp.uniform(i, (n,), dtype=nd), hp.uniform(100 + i, (n,), dtype=nd)
        ref.append(w - np.float32(0.5) * dw)
        o, kp = hp.optim_args(pkg, "fp32", w, dw, None, None, 0.5, 0.0)
        opts.append(o)
        keep.append((kp, w))
    table = (type(opts[0]) * len(opts))(*opts)
    assert gpu.ptl_gradient_descent_fp32_multi(table, len(opts)) == 0, gpu.ptl_last_error().decode()
    for (_, w), r in zip(keep, ref):
        assert np.allclose(w, r, rtol=0, atol=1e-6)


def test_a_rejected_step_returns_nothing_and_the_other_still_runs(pkg, gpu):
    """A stride that does not divide the extent: the weight gradient rejects it, the input gradient does not."""
    Ci, Co, H, K, s = 4, 8, 10, 3, 2
    Ho = hp.conv_out(H, K, 1, 1, s)
    x, w, dy = (hp.uniform(9 + i, sh) for i, sh in enumerate(((Ci, H, H), (Co, Ci, K, K), (Co, Ho, Ho))))
    dx, dw = np.full_like(x, 3), np.full_like(w, 3)
    a, keep = hp.conv2d_args(pkg, x, dx, w, dw, np.zeros_like(dy), dy, Ci, H, H, Co, K, K, Ho, Ho, (1, 1, 1, 1), (s, s))
    with pytest.raises(RuntimeError):
        pkg.call("pulp_conv2d_fp32_bw_cl", a)
    ref = torch.nn.grad.conv2d_input((1, Ci, H, H), torch.from_numpy(w).double(), torch.from_numpy(dy).double()[None],
                                     stride=s, padding=1)[0]
    assert np.all(dw == 3) and hp.rel_l2(dx, ref.numpy()) <= 1e-4


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("layer", ["linear", "conv2d", "conv2d_any"])
@pytest.mark.parametrize("place", ["host", "device"])
def test_a_step_without_a_buffer_leaves_the_other_one(pkg, gpu, dt, layer, place):
    """A gradient's buffer (or the input that the weight gradient reads) is missing: the call fails, and the step that has
    all of its tensors has run."""
    nd = hp.np_dtype(dt)
    n_in, n_out, Ci, Co, H = 24, 17, 16, 8, 8
    conv = layer != "linear"
    if layer == "conv2d_any":  # (the layer that the products with patch matrices take)
        Ci, Co, H = 24, 40, 21
    sh = ((Ci, H, H), (Co, Ci, 3, 3), (Co, H, H)) if conv else ((n_in,), (n_out, n_in), (n_out,))
    x, w, dy = (hp.uniform(20 + i, s, dtype=nd) for i, s in enumerate(sh))
    put = (lambda v: v.copy()) if place == "host" else (lambda v: torch.from_numpy(v).to(DEV))
    get = lambda v: v if isinstance(v, np.ndarray) else v.cpu().numpy()

    def run(missing):
        tx, tdx, tw, tdw, ty, tdy = (put(v) for v in (x, np.full(sh[0], 3, nd), w, np.full(sh[1], 3, nd), np.zeros(sh[2], nd), dy))
        if missing == "x":
            tx = None
        if missing == "dw":
            tdw = None
        if missing == "dx":
            tdx = None
        if conv:
            a, keep = hp.conv2d_args(pkg, tx, tdx, tw, tdw, ty, tdy, Ci, H, H, Co, 3, 3, H, H, pad=(1, 1, 1, 1))
        else:
            a, keep = hp.linear_args(pkg, tx, tdx, tw, tdw, ty, tdy, n_in, n_out)
        gpu.ptl_set_gemm_path(7 if layer == "conv2d_any" else 0)
        try:
            if missing:
                with pytest.raises(RuntimeError):
                    pkg.call("pulp_%s_%s_bw_cl" % ("conv2d" if conv else "linear", dt), a)
            else:
                pkg.call("pulp_%s_%s_bw_cl" % ("conv2d" if conv else "linear", dt), a)
        finally:
            gpu.ptl_set_gemm_path(0)
        assert gpu.ptl_sync() == 0
        return [None if t is None else get(t) for t in (tdx, tdw)]

    dx, dw = run("")
    for missing in ("x", "dw"):
        got = run(missing)
        assert hp.rel_l2(got[0], dx) <= (1e-3 if dt == "fp16" else 1e-5)
        assert got[1] is None or np.all(got[1] == 3)
    assert hp.rel_l2(run("dx")[1], dw) <= (1e-3 if dt == "fp16" else 1e-5)


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("place", ["host", "device"])
# dense layers: one sample, a batch on whole tiles, one on none; convolutions: small, wide, with patch matrices
@pytest.mark.parametrize("layer,ns,Ci,Co,H", [("linear", 1, 300, 5000, 0), ("linear", 64, 256, 256, 0), ("linear", 33, 127, 65, 0),
                                              ("conv2d", 1, 16, 32, 32), ("conv2d", 8, 64, 64, 16), ("conv2d", 5, 40, 130, 21)])
def test_an_input_gradient_written_over_the_input(pkg, gpu, dt, place, layer, ns, Ci, Co, H):
    """The weight gradient still is that of the input."""
    nd = hp.np_dtype(dt)
    conv = layer == "conv2d"
    sh = ((ns, Ci, H, H), (Co, Ci, 3, 3), (ns, Co, H, H)) if conv else ((ns, Ci), (Co, Ci), (ns, Co))
    x, w, dy = (hp.uniform(30 + i, s, dtype=nd) for i, s in enumerate(sh))
    put = (lambda v: v.copy()) if place == "host" else (lambda v: torch.from_numpy(v).to(DEV))
    get = lambda v: v if isinstance(v, np.ndarray) else v.cpu().numpy()
    res = []
    for alias in (0, 1):
        tx, tw, tdw, ty, tdy = (put(v) for v in (x, w, np.full(sh[1], 3, nd), np.zeros(sh[2], nd), dy))
        tdx = tx if alias else put(np.full(sh[0], 3, nd))
        if conv:
            a, keep = hp.conv2d_args(pkg, tx, tdx, tw, tdw, ty, tdy, Ci, H, H, Co, 3, 3, H, H, pad=(1, 1, 1, 1))
        else:
            a, keep = hp.linear_args(pkg, tx, tdx, tw, tdw, ty, tdy, Ci, Co)
        if ns == 1:
            pkg.call("pulp_%s_%s_bw_cl" % (layer, dt), a)
        else:
            pkg.call("ptl_%s_%s_bw_batched" % (layer, dt), a, ns)
        assert gpu.ptl_sync() == 0
        res.append([get(tdx), get(tdw)])
    for got, want in zip(res[1], res[0]):
        assert hp.rel_l2(got, want) <= (1e-3 if dt == "fp16" else 1e-5)


# (small tensors, which share a block; one with a block of its own)
@pytest.mark.parametrize("Ci,Co,P", [(12, 20, 35), (700, 600, 9)])
def test_a_step_reads_what_the_step_before_it_wrote(pkg, gpu, Ci, Co, P):
    """The weight gradient written over the weights: the input gradient is formed with it, on the host as on the device."""
    x, w, dy = (hp.uniform(40 + i, s) for i, s in enumerate(((Ci, P), (Co, Ci), (Co, P))))
    res = []
    for put in (lambda v: v.copy(), lambda v: torch.from_numpy(v).to(DEV)):
        tx, tdx, tw, ty, tdy = (put(v) for v in (x, np.zeros_like(x), w, np.zeros_like(dy), dy))
        a, keep = hp.pw_args(pkg, tx, tdx, tw, tw, ty, tdy, Ci, Co, 1, P)
        pkg.call("pulp_conv_pw_fp32_bw_cl", a)
        assert gpu.ptl_sync() == 0
        res.append([v if isinstance(v, np.ndarray) else v.cpu().numpy() for v in (tdx, tw)])
    dw = dy.astype(np.float64) @ x.T.astype(np.float64)
    assert hp.rel_l2(res[0][1], dw) <= 1e-5 and hp.rel_l2(res[0][0], dw.T @ dy) <= 1e-5
    for h, d in zip(*res):
        assert np.array_equal(h, d)


# (two parts and an odd end; the largest tensor with a block of its own: 32 MiB; one row beyond)
@pytest.mark.parametrize("n_in,n_out", [(525, 1001), (2896, 2896), (2897, 2897)])
def test_large_host_tensors_travel_in_parts(pkg, gpu, n_in, n_out):
    res = []
    for place in (lambda a: a.copy(), lambda a: torch.from_numpy(a).to(DEV)):
        t = [place(a) for a in (hp.uniform(1, (n_in,)), np.zeros(n_in, np.float32), hp.uniform(2, (n_out, n_in)),
                                np.full((n_out, n_in), 3, np.float32), np.zeros(n_out, np.float32), hp.uniform(3, (n_out,)))]
        a, keep = hp.linear_args(pkg, *t, n_in, n_out)
        pkg.call("pulp_linear_fp32_fw_cl", a)
        pkg.call("pulp_linear_fp32_bw_cl", a)
        assert gpu.ptl_sync() == 0
        res.append([v if isinstance(v, np.ndarray) else v.cpu().numpy() for v in t])
    for h, d in zip(*res):
        assert np.array_equal(h, d)


# (layers that the route of both gradients in one launch takes, and ones that it is asked for and leaves to the two steps: few
# channels, channel-minor; the last one's tensors are a transfer each)
@pytest.mark.parametrize("dt,ns,Ci,Co,H,K,s,copies", [("fp16", 4, 24, 48, 29, 1, 1, 2), ("fp32", 2, 9, 8, 12, 3, 1, 2), ("fp16", 4, 3, 48, 29, 1, 1, 2),
                                                      ("fp16", 4, 4, 93, 15, 3, 2, 2), ("fp16", 4, 3, 64, 181, 1, 1, 3)])
def test_a_backward_call_fetches_a_host_tensor_once(pkg, gpu, dt, ns, Ci, Co, H, K, s, copies):
    nd, p = hp.np_dtype(dt), K // 2
    Ho = hp.conv_out(H, K, p, p, s)
    x, w, dy = (hp.uniform(31 + i, sh, dtype=nd) for i, sh in enumerate(((ns, H, H, Ci), (Co, K, K, Ci), (ns, Ho, Ho, Co))))
    res = []
    for place in (lambda a: a.copy(), lambda a: torch.from_numpy(a).to(DEV)):
        t = [place(a) for a in (x, np.full_like(x, 3), w, np.full_like(w, 3), np.zeros_like(dy), dy)]
        a, keep = hp.conv2d_args(pkg, *t, Ci, H, H, Co, K, K, Ho, Ho, (p,) * 4, (s, s), hwc=1)
        before = gpu.ptl_staging_copies()
        pkg.call("ptl_conv2d_%s_bw_batched" % dt, a, ns)
        assert gpu.ptl_sync() == 0
        assert gpu.ptl_staging_copies() - before == (0 if res else copies)
        res.append([v if isinstance(v, np.ndarray) else v.cpu().numpy() for v in t])
    for h, d in zip(*res):
        assert np.array_equal(h, d)
