"""Outcomes and states of noisy lists applied as runs, in single precision too:
a run may differ from the same operations one by one in a draw within rounding
of its boundary, and in nothing else."""
import numpy as np
import pytest

from refcirc import random_spec, to_bt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [("c64", 2e-5), ("c128", 1e-11)])
@pytest.mark.parametrize("N", [4, 9, 13])
def test_outcomes_over_many_seeds(bt, N, prec, tol):
    """40 lists of 50 operations, about 40 draws each.  FP32 probabilities are
    off by some 1e-6 at most, so a draw meets its boundary in 1 of 25000 lists
    or fewer: one list may, two do not.  complex128 agrees throughout."""
    noise = bt.NoiseModel("depolarizing", 0.05, "amplitude_damping", 0.1)
    other = 0
    for seed in range(40):
        ops = to_bt(random_spec(N, 50, np.random.default_rng(1000 * N + seed)), bt)
        a, b = bt.zero_state(N, prec), bt.zero_state(N, prec)
        ra, rb = bt.UniformStream(seed, 2), bt.UniformStream(seed, 2)
        oa = bt.apply(a, ops, noise=noise, track_measurements=True, rng=ra)[1]
        ob = []
        for o in ops:
            ob += bt.apply(b, o, noise=noise, track_measurements=True, rng=rb)[1]
        assert len(oa) == len(ob)
        x, y = a.to_numpy(), b.to_numpy()
        if oa != ob or ra.draw != rb.draw:
            other += 1
            continue
        if np.isnan(x).any() or np.isnan(y).any():
            assert np.array_equal(np.isnan(x), np.isnan(y))
            continue
        if np.abs(x - y).max() > tol:  # a channel's draw, which leaves no outcome
            other += 1
    assert other <= (1 if prec == "c64" else 0)
