"""Calls that have another way when the workspace cannot grow during a capture: they take it, their results hold, the workspace stays as it
is and no error is left behind.  Each case in a process of its own, whose workspace is as small as it is reserved."""
import ctypes
import os
import subprocess
import sys

import pytest
import torch

import helpers as hp

pytestmark = pytest.mark.gpu
ROOM = 8 << 20


def sizes(gpu):
    ws, sc = ctypes.c_size_t(0), ctypes.c_size_t(0)
    gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
    return ws.value


def replayed(gpu, call, fresh, room):
    """`call` in a graph that is replayed three times, each time onto `fresh`ly filled results."""
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    gpu.ptl_set_stream(ctypes.c_void_p(side.cuda_stream))
    with torch.cuda.graph(graph, stream=side):
        rc = call()
    assert (rc, gpu.ptl_last_error()) == (0, b"") and sizes(gpu) == room, (rc, gpu.ptl_last_error(), sizes(gpu))
    for _ in range(3):
        fresh()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
    gpu.ptl_set_stream(None)
    return graph


def attention(pkg, gpu, case):
    from test_gpu_attention_parts import backward

    def check(data, diff):
        x, dy, att = data["x"].double(), diff["y"].double(), data["att"].double()
        flat = lambda t: t.transpose(0, 1).reshape(t.shape[1], -1)
        rel = lambda got, ref: float((got.double() - ref).norm() / ref.norm())
        for w, n in (("wq", "q"), ("wk", "k"), ("wv", "v")):  # (32-bit sums of sums of 32: 2e-7 in the mean)
            assert rel(diff[w], flat(diff[n].double()) @ flat(x).T.contiguous()) <= 1e-6, w
        assert rel(diff["wo"].reshape(diff["y"].shape[1], -1), flat(dy) @ flat(att).T.contiguous()) <= 1e-6

    def run(call, diff):
        run.graph = replayed(gpu, call, lambda: [t.zero_() for n, t in diff.items() if n != "y"], ROOM)

    assert gpu.ptl_reserve(1, ROOM) == 0 and sizes(gpu) == ROOM
    check(*backward(pkg, gpu, *case, run=run))
    check(*backward(pkg, gpu, *case))
    assert sizes(gpu) > ROOM  # (a call that may grow it has other parts)


def one_sample(pkg, gpu, case):
    n_in, n_out = case
    g = torch.Generator().manual_seed(1)
    x, w, dy = ((torch.rand(s, generator=g) - 0.5).cuda() for s in ((1, n_in), (n_out, n_in), (1, n_out)))
    dx, dw = torch.empty_like(x), torch.empty_like(w)
    a, keep = hp.linear_args(pkg, x, dx, w, dw, dy, dy, n_in, n_out)
    call = lambda: gpu.ptl_linear_fp32_bw_batched(ctypes.byref(a), 1)
    ref = dy.double() @ w.double()

    def check():
        assert torch.equal(dw, dy.t() * x) and float((dx.double() - ref).norm() / ref.norm()) <= 1e-6

    assert sizes(gpu) == 0
    graph = replayed(gpu, call, lambda: [t.fill_(7) for t in (dx, dw)], 0)
    check()
    assert call() == 0 and gpu.ptl_sync() == 0 and sizes(gpu) > 0
    check()


def in_a_process(what, case):
    import __graft_entry__ as ge
    pkg = ge.load_package()
    gpu = pkg.load()
    assert gpu.ptl_init(0) == 0
    globals()[what](pkg, gpu, case)
    print("finished", flush=True)


# samples, tokens, token size, features, heads: parts that the first plan cannot have (22 MiB); a first plan that needs no workspace
# (parts of 200 slabs, the whole contraction) and is cut again (20 MiB).  One sample: inputs, outputs
@pytest.mark.parametrize("what,case", [("attention", (28, 130, 384, 384, 12)), ("attention", (40, 140, 512, 512, 8)), ("one_sample", (64, 16384))])
def test_captured(gpu, what, case):
    here = os.path.dirname(os.path.abspath(__file__))
    code = "import sys; sys.path[:0] = [%r, %r]; import test_gpu_refused_growth as t; t.in_a_process(%r, %r)" % (here, os.path.dirname(here), what, case)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "finished" in r.stdout, r.stdout + r.stderr
