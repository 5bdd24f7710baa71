"""The parts that the weight gradients of attention are formed in beside the input gradient: against 64 bits where a part is a few
slabs, where there are several rounds of workgroups and where nothing is split; and with a workspace too small for them, in a
capture that must not grow it."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu


def backward(pkg, gpu, ns, L, E, F, heads, run=None):
    """Backward from random states; (arguments' tensors, gradients), the gradients of `run` if that calls it."""
    sh = hp.mhsa_shapes(ns, L, E, F, heads)
    g = torch.Generator().manual_seed(L + F)
    data = {n: (torch.rand(s, generator=g) - 0.5).cuda() for n, s in sh.items()}
    data["p"] /= L
    diff = {n: torch.full(sh[n], 7.0, device="cuda") for n in ("q", "k", "v", "att", "p", "wo")}
    diff.update({n: torch.full((F, E), 7.0, device="cuda") for n in ("wq", "wk", "wv")})
    diff["x"], diff["y"] = torch.zeros(sh["x"], device="cuda"), (torch.rand(sh["y"], generator=g) - 0.5).cuda()
    a, keep = hp.mhsa_args(pkg, data, diff, L, E, F, heads)
    call = lambda: gpu.ptl_mhsa_fp32_bw_batched(ctypes.byref(a), ns)
    if run:
        run(call, diff)
    else:
        assert call() == 0, gpu.ptl_last_error().decode()
        assert gpu.ptl_sync() == 0
    return data, diff


# samples, tokens, token size, features, heads
@pytest.mark.parametrize("case", [(1, 5, 8, 8, 1), (64, 17, 192, 192, 3), (40, 33, 70, 96, 2), (31, 128, 64, 64, 2), (12, 131, 192, 192, 3),
                                  (8, 130, 320, 320, 10), (64, 129, 64, 128, 2), (33, 192, 192, 192, 6)])
def test_against_64_bits(pkg, gpu, case):
    ns, L, E, F, heads = case
    data, diff = backward(pkg, gpu, ns, L, E, F, heads)
    x, dy, att = data["x"].double(), diff["y"].double(), data["att"].double()
    flat = lambda t: t.transpose(0, 1).reshape(t.shape[1], -1)  # [rows][samples x tokens]
    rel = lambda got, ref: float((got.double() - ref).norm() / ref.norm())
    for w, n in (("wq", "q"), ("wk", "k"), ("wv", "v")):
        assert rel(diff[w], flat(diff[n].double()) @ flat(x).T) <= 1e-6, w  # (32-bit sums of sums of 32: 2e-7 in the mean)
    assert rel(diff["wo"].reshape(E, F), flat(dy) @ flat(att).T) <= 1e-6
    dx = sum(data[w].double().reshape(E, F) @ flat(diff[n].double()) for w, n in (("wq", "q"), ("wk", "k"), ("wv", "v")))
    assert rel(flat(diff["x"]), dx) <= 1e-6


# More than 128 tokens and parts of sixteen slabs (32 where a CU would have three workgroups): as bf16 pieces; fewer, or 128 tokens: not
@pytest.mark.parametrize("case,form", [((32, 197, 192, 192, 3), 1), ((64, 130, 70, 96, 2), 1), ((2, 256, 512, 512, 8), 1), ((64, 147, 192, 192, 4), 1), ((64, 192, 192, 192, 3), 1),
                                       ((8, 256, 384, 384, 8), 0), ((16, 131, 512, 512, 8), 0), ((64, 128, 192, 192, 3), 0)])
def test_weight_gradients_in_pieces(pkg, gpu, case, form):
    test_against_64_bits(pkg, gpu, case)
    assert gpu.ptl_last_gemm_form() == form


SMALL = (28, 130, 384, 384, 12)  # 22 MiB of partial sums; a fifth of the parts fit in 8


def captured_in_a_small_workspace():
    import __graft_entry__ as ge
    pkg = ge.load_package()
    gpu = pkg.load()
    assert gpu.ptl_init(0) == 0 and gpu.ptl_reserve(1, 8 << 20) == 0
    ws, sc = ctypes.c_size_t(0), ctypes.c_size_t(0)
    gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
    assert ws.value == 8 << 20, ws.value
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()

    def run(call, diff):
        torch.cuda.synchronize()
        gpu.ptl_set_stream(ctypes.c_void_p(side.cuda_stream))
        with torch.cuda.graph(graph, stream=side):
            rc = call()
        assert rc == 0, gpu.ptl_last_error().decode()
        for _ in range(3):
            for n, t in diff.items():
                if n != "y":
                    t.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()

    _, got = backward(pkg, gpu, *SMALL, run=run)
    gpu.ptl_set_stream(None)
    gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
    assert ws.value == 8 << 20, ws.value
    _, ref = backward(pkg, gpu, *SMALL)
    gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
    assert ws.value > 8 << 20, ws.value  # the parts that a call takes that may grow it
    for n in ("wq", "wk", "wv", "wo", "x", "q", "k", "v"):
        assert float((got[n].double() - ref[n].double()).norm() / ref[n].double().norm()) <= 1e-6, n
    print("captured", flush=True)


def test_capture_with_a_small_workspace(gpu):
    here = os.path.dirname(os.path.abspath(__file__))
    code = "import sys; sys.path[:0] = [%r, %r]; import test_gpu_attention_parts as t; t.captured_in_a_small_workspace()" % (here, os.path.dirname(here))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "captured" in r.stdout, r.stdout + r.stderr


def large_step():
    import __graft_entry__ as ge
    pkg = ge.load_package()
    gpu = pkg.load()
    assert gpu.ptl_init(0) == 0
    ws, sc = ctypes.c_size_t(0), ctypes.c_size_t(0)
    for case in ((64, 256, 512, 512, 8), (64, 256, 1024, 1024, 16)):
        test_against_64_bits(pkg, gpu, case)
        gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
        print(case, ws.value >> 20, "MiB", flush=True)
        assert 0 < ws.value <= 160 << 20, ws.value
    print("bounded", flush=True)


def test_workspace_of_large_steps(gpu):
    """52 and 64 MiB of partial sums (the latter 208 in parts of 40 slabs), and the quarter more that is allocated."""
    here = os.path.dirname(os.path.abspath(__file__))
    code = "import sys; sys.path[:0] = [%r, %r]; import test_gpu_attention_parts as t; t.large_step()" % (here, os.path.dirname(here))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "bounded" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("what", ["infinity", "nan", "huge", "tiny"])
@pytest.mark.parametrize("case", [(64, 130, 70, 96, 2), (32, 197, 192, 192, 3)])
def test_values_outside_the_range_of_the_pieces(pkg, gpu, case, what):
    """In the tokens and in the attention map, which only the weight gradients read: in pieces beside an input gradient that is not, which
    keeps its bits.  Features without such a value keep theirs in the tiles that have none."""
    ns, L, E, F, heads = case
    sh = hp.mhsa_shapes(ns, L, E, F, heads)
    g = torch.Generator().manual_seed(L)
    data = {n: (torch.rand(s, generator=g) - 0.5).cuda() for n, s in sh.items()}
    data["p"] /= L
    dy = (torch.rand(sh["y"], generator=g) - 0.5).cuda()

    def run():
        diff = {n: torch.full(sh[n], 7.0, device="cuda") for n in ("q", "k", "v", "att", "p", "wo")}
        diff.update({n: torch.full((F, E), 7.0, device="cuda") for n in ("wq", "wk", "wv")})
        diff["x"], diff["y"] = torch.zeros(sh["x"], device="cuda"), dy
        a, keep = hp.mhsa_args(pkg, data, diff, L, E, F, heads)
        assert gpu.ptl_mhsa_fp32_bw_batched(ctypes.byref(a), ns) == 0, gpu.ptl_last_error().decode()
        assert gpu.ptl_sync() == 0 and gpu.ptl_last_gemm_form() == 1
        return diff

    plain = run()
    if what == "tiny":  # (the third piece of 1e-35 would lie below the smallest bf16)
        data["x"].mul_(1e-35)
        data["att"].mul_(1e-35)
    else:  # (huge: rounds up to infinity as a bf16)
        value = {"infinity": float("inf"), "nan": float("nan"), "huge": 3.4e38}[what]
        data["x"][ns // 2, 66, 77] = value
        data["att"][1, 67, 5] = -value
    diff = run()
    for n in ("x", "q", "k", "v", "att"):
        assert torch.equal(diff[n], plain[n]), n
    flat = lambda t: t.double().transpose(0, 1).reshape(t.shape[1], -1)
    for w, left, right in (("wq", diff["q"], data["x"]), ("wk", diff["k"], data["x"]), ("wv", diff["v"], data["x"]), ("wo", dy, data["att"])):
        if what in ("infinity", "nan"):
            assert torch.equal(diff[w].reshape(left.shape[1], -1)[:, :64], plain[w].reshape(left.shape[1], -1)[:, :64]), w
        ref, got = flat(left) @ flat(right).T.contiguous(), diff[w].reshape(left.shape[1], -1).double()
        ref = torch.where(ref.abs() > torch.finfo(torch.float32).max, ref * float("inf"), ref)
        assert torch.equal(got.isnan(), ref.isnan()), w
        assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[ref.isinf()], ref[ref.isinf()]), w
        fin = ref.isfinite()
        size = ref[fin].abs().max() if what == "huge" else (ref[fin] ** 2).mean().sqrt()
        # up to 8320 products, 320 slabs: sqrt(320 / 3) roundings of 2^-25 and of 2^-24 in eight, six times that for the largest of 37 000
        assert float((got[fin] - ref[fin]).abs().max()) <= 4e-6 * float(size), w
