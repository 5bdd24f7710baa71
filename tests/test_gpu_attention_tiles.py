"""Attention steps at the edges of the score tiles (32 queries, groups of eight keys, 256 tokens), of the head blocks (32, 64)
and of the projections' pieces, against the CPU oracle."""
import numpy as np
import pytest

import helpers as hp
from test_gpu_mhsa import BW_OUT, FW_OUT, TOL, gpu_step, oracle_step

pytestmark = pytest.mark.gpu


# samples, tokens, token size, features, heads
@pytest.mark.parametrize("case", [
    (2, 4, 4, 4, 1), (1, 3, 8, 6, 2), (2, 8, 5, 33, 1), (3, 31, 36, 64, 2), (1, 32, 20, 32, 1), (9, 33, 70, 62, 2),
    (1, 129, 33, 96, 3), (2, 201, 12, 48, 1), (1, 255, 16, 64, 1), (1, 256, 8, 128, 2), (1, 257, 8, 64, 1)])
def test_step(pkg, orc, gpu, case):
    ns, L, E, F, heads = case
    d, dy = hp.mhsa_inputs(L * 131 + F, ns, L, E, F, heads)
    x0 = hp.uniform(L + 7, (ns, E, L))
    ref_data, ref_diff = oracle_step(pkg, orc, d, dy, x0, ns, L, E, F, heads)
    got_data, got_diff = gpu_step(pkg, gpu, d, dy, x0, ref_data, ns, L, E, F, heads, True, named=False)
    for n in FW_OUT:
        assert hp.rel_l2(got_data[n], ref_data[n]) <= TOL, "forward %s" % n
    for n in BW_OUT:
        assert hp.rel_l2(got_diff[n], ref_diff[n]) <= TOL, "backward %s" % n


def test_a_sample_is_the_same_in_every_batch(pkg, orc, gpu):
    """Few samples are formed in quarters of the tiles that a batch takes, in the same order of summation."""
    ns, L, E, F, heads = 96, 133, 40, 64, 2
    d, dy = hp.mhsa_inputs(0x5A3E, ns, L, E, F, heads)
    x0 = np.zeros((ns, E, L), np.float32)
    state = {n: np.zeros(s, np.float32) for n, s in hp.mhsa_shapes(ns, L, E, F, heads).items() if n in FW_OUT}
    rng = np.random.default_rng(7)
    for n in state:  # (the backward pass starts from these, whatever they are)
        state[n][...] = rng.random(state[n].shape, np.float32) / (L if n == "p" else 1)
    full_d, full_g = gpu_step(pkg, gpu, d, dy, x0, state, ns, L, E, F, heads, True, named=False)
    for b in (0, 95):
        db = dict(d)
        db["x"] = d["x"][b:b + 1]
        one_d, one_g = gpu_step(pkg, gpu, db, dy[b:b + 1], x0[b:b + 1], {n: state[n][b:b + 1] for n in FW_OUT}, 1, L, E, F,
                                heads, True, named=False)
        for n in FW_OUT:
            assert np.array_equal(one_d[n][0], full_d[n][b]), (b, n)
        for n in ("att", "p", "q", "k", "v", "x"):
            assert np.array_equal(one_g[n][0], full_g[n][b]), (b, n)
