"""A growth of the library's workspace that is refused during a capture leaves the workspace that is there."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_a_refused_growth_keeps_the_workspace(pkg, gpu):
    assert gpu.ptl_reserve(1 << 20, 0) == 0, gpu.ptl_last_error().decode()
    ws, sc = ctypes.c_size_t(0), ctypes.c_size_t(0)
    gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
    have = ws.value
    src, dst = torch.rand(16, device="cuda"), torch.zeros(16, device="cuda")
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    gpu.ptl_set_stream(ctypes.c_void_p(side.cuda_stream))
    try:
        with torch.cuda.graph(graph, stream=side):
            refused = gpu.ptl_reserve(have + 1, 0)
            kept = gpu.ptl_reserve(1, 0)
            copied = gpu.ptl_copy_bytes(ctypes.c_void_p(src.data_ptr()), ctypes.c_void_p(dst.data_ptr()), 64)
    finally:
        gpu.ptl_set_stream(None)
    assert (refused, kept, copied) == (2, 0, 0), gpu.ptl_last_error().decode()
    gpu.ptl_reserved(ctypes.byref(ws), ctypes.byref(sc))
    assert ws.value == have
    assert gpu.ptl_reserve(1, 0) == 0, gpu.ptl_last_error().decode()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(src, dst)
