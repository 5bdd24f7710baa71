"""The per-head attention kernels where a head's block of q, k, v or the attention map's gradient comes in aligned pieces of 16
bytes (odd numbers of tokens, heads of whole fours) and where it does not (a buffer one element off): the same bits, and those
of the CPU oracle.  Rows follow each other there, so that what lies beyond a row's end is the next row: with infinities in
one feature, the others keep their bits."""
import ctypes

import numpy as np
import pytest
import torch

import helpers as hp
from test_gpu_mhsa import FW_OUT, TOL, oracle_step

pytestmark = pytest.mark.gpu


def step(pkg, gpu, d, dy, state, ns, L, E, F, heads, off):
    """Forward from the inputs, backward from `state`; the activations start `off` elements behind a 16-byte boundary."""
    sh = hp.mhsa_shapes(ns, L, E, F, heads)

    def at(z):
        flat = torch.empty(z.size + off, device="cuda")
        flat[off:] = torch.from_numpy(np.ascontiguousarray(z).reshape(-1)).cuda()
        return flat[off:].view(z.shape)

    empty = lambda n, s=None: at(np.full(s or sh[n], 7.0, np.float32))
    data = {n: at(v) for n, v in d.items()}
    data.update({n: empty(n) for n in FW_OUT})
    a, keep = hp.mhsa_args(pkg, data, {}, L, E, F, heads)
    assert gpu.ptl_mhsa_fp32_fw_batched(ctypes.byref(a), ns) == 0, gpu.ptl_last_error().decode()
    given = {n: at(v) for n, v in d.items()}
    given.update({n: at(state[n]) for n in FW_OUT})
    diff = {n: empty(n) for n in ("q", "k", "v", "att", "p", "wo")}
    diff.update({n: empty(n, (F, E)) for n in ("wq", "wk", "wv")})
    diff["x"], diff["y"] = at(np.zeros(sh["x"], np.float32)), at(dy)
    b, keep2 = hp.mhsa_args(pkg, given, diff, L, E, F, heads)
    assert gpu.ptl_mhsa_fp32_bw_batched(ctypes.byref(b), ns) == 0, gpu.ptl_last_error().decode()
    assert gpu.ptl_sync() == 0
    return {n: data[n].cpu().numpy() for n in FW_OUT}, {n: diff[n].cpu().numpy() for n in ("att", "p", "q", "k", "v")}


# samples, tokens, features, heads: 1 to 3 tokens beyond whole fours, groups of eight and tiles of 32; heads at the ends of both
# sizes of block, one of them of no whole fours; 128 and 129 tokens (blocks of features per wave); both ends of the range
@pytest.mark.parametrize("case", [(2, 5, 8, 2), (1, 31, 4, 1), (2, 33, 72, 2), (1, 127, 64, 2), (2, 129, 64, 1), (1, 130, 96, 2),
                                  (1, 131, 66, 2), (1, 128, 48, 1), (1, 132, 120, 2), (2, 197, 64, 1), (1, 250, 32, 1),
                                  (1, 255, 120, 2), (1, 256, 64, 2)])
def test_aligned_or_not(pkg, orc, gpu, case):
    ns, L, F, heads = case
    E, H = 20, F // heads
    d, dy = hp.mhsa_inputs(L * 31 + F, ns, L, E, F, heads)
    ref_d, ref_g = oracle_step(pkg, orc, d, dy, np.zeros((ns, E, L), np.float32), ns, L, E, F, heads)
    fw, bw = step(pkg, gpu, d, dy, ref_d, ns, L, E, F, heads, 0)
    for n in FW_OUT:
        assert hp.rel_l2(fw[n], ref_d[n]) <= TOL, n
    for n in bw:
        assert hp.rel_l2(bw[n], ref_g[n]) <= TOL, n
    fw1, bw1 = step(pkg, gpu, d, dy, ref_d, ns, L, E, F, heads, 1)
    for n in ("p", "att"):
        assert np.array_equal(fw[n], fw1[n]), n
    for n in bw:
        assert np.array_equal(bw[n], bw1[n]), n

    # one feature of the first head infinite: v in the forward pass; k, q and then the map's gradient in the backward one
    rest = np.arange(F) != 1
    poisoned = dict(d, bv=np.where(rest, d["bv"], np.inf).astype(np.float32))
    state = dict(ref_d, k=ref_d["k"].copy(), q=ref_d["q"].copy())
    state["k"][:, 1] = state["q"][:, 1] = np.inf
    fw2, bw2 = step(pkg, gpu, poisoned, dy, state, ns, L, E, F, heads, 0)
    assert np.array_equal(fw2["att"][:, rest], fw["att"][:, rest])
    for n in ("q", "k", "v"):
        assert np.array_equal(bw2[n][:, rest], bw[n][:, rest]), n
    poisoned = dict(d, wo=d["wo"].copy())
    poisoned["wo"].reshape(E, F)[:, 1] = np.inf
    _, bw3 = step(pkg, gpu, poisoned, dy, ref_d, ns, L, E, F, heads, 0)
    assert np.array_equal(bw3["v"][:, rest], bw["v"][:, rest])
    assert np.array_equal(bw3["q"][:, H:], bw["q"][:, H:]) and np.array_equal(bw3["k"][:, H:], bw["k"][:, H:])
