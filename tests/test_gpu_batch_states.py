"""Batches with their final states: reductions finished inside the pass
launch (one workgroup per state, a few, many) and states exported through the
staging (many states per launch, a state larger than the staging, a basis
state never written) against the same trajectories run one at a time, whose
parity with the oracle is tested elsewhere.

Tolerances: the same bounds as the trajectory executors' (complex128 1e-12,
complex64 1e-5, largest amplitude error), doubled for the two runs' rounding."""
import numpy as np
import pytest

from refcirc import random_spec, to_bt

pytestmark = pytest.mark.gpu
TOL = {"c64": 2e-5, "c128": 2e-12}
KINDS = ("gate1", "gate2", "chan1", "chan2", "meas", "reset")
NM = ("depolarizing", 0.02, "amplitude_damping", 0.1)


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N,nops,ntraj", [(1, 12, 70), (3, 30, 33), (12, 60, 40), (14, 80, 160), (17, 60, 17),
                                           (21, 40, 3), (23, 30, 2)])
def test_batch_matches_single_runs(bt, N, nops, ntraj, prec):
    from bluetangle_jl_amd.circuit import Circuit
    from bluetangle_jl_amd.core import StateVector
    kinds = KINDS if N > 1 else ("gate1", "chan1", "meas", "reset")
    if N >= 3:
        kinds += ("kraus",)  # up to three bits: the widest reductions
    spec = random_spec(N, nops, np.random.default_rng(100 * N + nops), kinds=kinds)
    c = Circuit(to_bt(spec, bt), N, bt.NoiseModel(*NM))
    outs, states, st = c.run_batch(ntraj, seed=9, prec=prec, keep_states=True)
    again, states2, _ = c.run_batch(ntraj, seed=9, prec=prec, keep_states=True)
    assert again == outs and np.array_equal(states, states2, equal_nan=True)  # fixed order: bit for bit
    some, other = range(0, ntraj, max(1, ntraj // 12)), 0
    for t in some:
        s = StateVector(N, prec)
        o, _ = c.run_on(s, seed=9, traj=t)
        if o != outs[t]:  # a draw within rounding of its boundary
            other += 1
            continue
        v = s.to_numpy()
        if np.isnan(v).any():  # a branch of probability 0, as in the oracle
            assert np.array_equal(np.isnan(v), np.isnan(states[t])), t
            continue
        assert np.abs(states[t] - v).max() < TOL[prec], t
    assert other <= (0 if prec == "c128" else 1)


def test_untouched_state(bt):
    """A circuit that leaves |0..0> as it is."""
    from bluetangle_jl_amd.circuit import Circuit
    c = Circuit([bt.Op("MZ", 1), bt.Op("MZ", 5)], 6, False)
    outs, states, _ = c.run_batch(9, seed=1, prec="c64", keep_states=True)
    want = np.zeros(64, dtype=complex)
    want[0] = 1.0
    assert all(o == [0, 0] for o in outs) and np.array_equal(states, np.tile(want, (9, 1)))
