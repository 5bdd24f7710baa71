"""Attention's projections over a batch whose tokens are no whole tiles: the columns of all samples follow each other, and a
tile holds those of two of them (33 and 65 tokens in tiles of 32, 129 and more in tiles of 64; pieces of four tokens end inside
a sample's last one)."""
import numpy as np
import pytest

import helpers as hp
from test_gpu_mhsa import FW_OUT, TOL, gpu_step, oracle_step

pytestmark = pytest.mark.gpu


# samples, tokens, token size, features, heads
@pytest.mark.parametrize("case", [(90, 33, 192, 192, 3), (60, 65, 70, 200, 4), (64, 129, 160, 192, 3), (52, 130, 197, 190, 5),
                                  (44, 197, 192, 192, 3)])
def test_first_and_last_sample(pkg, orc, gpu, case):
    ns, L, E, F, heads = case
    d, dy = hp.mhsa_inputs(L * 17 + F, ns, L, E, F, heads)
    x0 = hp.uniform(L + 3, (ns, E, L))
    state = {n: np.zeros(s, np.float32) for n, s in hp.mhsa_shapes(ns, L, E, F, heads).items() if n in FW_OUT}
    rng = np.random.default_rng(L)
    for n in state:  # (the backward pass starts from these, whatever they are)
        state[n][...] = rng.random(state[n].shape, np.float32) / (L if n == "p" else 1)
    full_d, full_g = gpu_step(pkg, gpu, d, dy, x0, state, ns, L, E, F, heads, True, named=False)
    for b in (0, ns - 1):  # one sample has no other behind it: the same bits
        db = dict(d, x=d["x"][b:b + 1])
        one_d, one_g = gpu_step(pkg, gpu, db, dy[b:b + 1], x0[b:b + 1], {n: state[n][b:b + 1] for n in FW_OUT}, 1, L, E, F,
                                heads, True, named=False)
        for n in FW_OUT:
            assert np.array_equal(one_d[n][0], full_d[n][b]), (b, n)
        for n in ("att", "p", "q", "k", "v", "x"):
            assert np.array_equal(one_g[n][0], full_g[n][b]), (b, n)
    two = dict(d, x=d["x"][-2:])
    ref_d, _ = oracle_step(pkg, orc, two, dy[-2:], x0[-2:], 2, L, E, F, heads)
    for n in FW_OUT:
        assert hp.rel_l2(full_d[n][-2:], ref_d[n]) <= TOL, n
