"""Lists of operations through apply: runs that go to bt_apply_ops against the
same list applied one operation at a time."""
import numpy as np
import pytest

from refcirc import random_spec, to_bt

pytestmark = pytest.mark.gpu
NM = ("depolarizing", 0.05, "amplitude_damping", 0.1)
TOL = {"c64": 2e-5, "c128": 1e-11}


def _state(bt, N, prec, seed, norm=1.0):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=2 ** N) + 1j * rng.normal(size=2 ** N)
    return bt.from_numpy(norm * v / np.linalg.norm(v), prec), norm * v / np.linalg.norm(v)


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("noisy", [False, True])
@pytest.mark.parametrize("N", [3, 8, 12, 14])
def test_list_matches_one_at_a_time(bt, N, noisy, prec):
    """Every op kind, an input state that is not normalised, and rng position:
    the same outcomes, the same state, the same draws consumed."""
    rng = np.random.default_rng(31 * N + noisy)
    spec = random_spec(N, 50, rng)
    noise = bt.NoiseModel(*NM) if noisy else False
    for norm in (1.0, 0.8):
        a, _ = _state(bt, N, prec, N, norm)
        b = a.copy()
        ra, rb = bt.UniformStream(5, 1), bt.UniformStream(5, 1)
        ops = to_bt(spec, bt)
        _, oa = bt.apply(a, ops, noise=noise, track_measurements=True, rng=ra)
        ob = []
        for o in ops:
            _, x = bt.apply(b, o, noise=noise, track_measurements=True, rng=rb)
            ob += x
        assert ra.draw == rb.draw
        x, y = a.to_numpy(), b.to_numpy()
        if oa != ob:  # a draw within rounding of its boundary
            assert prec == "c64"
            continue
        assert np.array_equal(np.isnan(x), np.isnan(y))
        assert np.nanmax(np.abs(x - y)) <= TOL[prec]


@pytest.mark.parametrize("prec,N", [("c64", 23), ("c128", 22)])
def test_short_runs_on_large_states(bt, prec, N):
    """From _RUN_LARGE bytes on four gates are a run: distant, adjacent and
    controlled ones, then back."""
    st = bt.zero_state(N, prec)
    ops = [bt.Op("H", 1), bt.Op("CNOT", 1, N), bt.Op("RY(0.7)", N // 2), bt.Op("RX(1.1)", 2, control=N // 2)]
    bt.apply(st, ops)
    ref = bt.zero_state(N, prec)
    for o in ops:
        bt.apply(ref, o)
    assert abs(st.inner(ref) - 1) <= (1e-6 if prec == "c64" else 1e-13)
    idx = [0, 1, 2 ** (N - 1), 2 ** (N - 1) + 1]
    assert np.abs(st.gather(idx) - ref.gather(idx)).max() <= (1e-6 if prec == "c64" else 1e-14)


def test_what_was_refused_is_refused_where_it_was(bt):
    """An op that raises in the middle of a list: the ones before it have been
    applied, the ones after it have not."""
    N = 4
    good = [bt.Op("H", 1 + i % N) for i in range(12)]
    for bad in (bt.Op("CNOT", 1, 9), "nonsense", bt.Op("RES", 9)):
        st = bt.zero_state(N, "c128")
        with pytest.raises(Exception):
            bt.apply(st, good[:11] + [bad] + good)
        ref = bt.zero_state(N, "c128")
        for o in good[:11]:
            bt.apply(ref, o)
        assert np.abs(st.to_numpy() - ref.to_numpy()).max() <= 1e-14
    # a noise model without a two-qubit channel
    st = bt.zero_state(N, "c128")
    with pytest.raises(ValueError):
        bt.apply(st, good + [bt.Op("CNOT", 1, 2)], noise=bt.NoiseModel(bt.Noise1("depolarizing", 0.0), False),
                 rng=bt.UniformStream(1))


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_a_state_without_a_norm(bt, prec):
    """Sampling on a zero state goes op by op, on the same draws."""
    N = 3
    ops = [bt.Op("H", 1 + i % N) for i in range(9)] + [bt.Op("MZ", 1), bt.Op("MR", 2)]
    out = []
    for one in (False, True):
        st = bt.zero_state(N, prec)
        st.upload(np.zeros(8))
        r = bt.UniformStream(3)
        outs = []
        if one:
            for o in ops:
                outs += bt.apply(st, o, track_measurements=True, rng=r)[1]
        else:
            outs = bt.apply(st, ops, track_measurements=True, rng=r)[1]
        out.append((outs, r.draw, st.to_numpy()))
    assert out[0][:2] == out[1][:2]
    assert np.array_equal(out[0][2], out[1][2], equal_nan=True)


def test_conditionals_and_functions_between_runs(bt):
    """ifOp and OpF end a run; the operations around them still apply in order."""
    N = 5
    ops = [bt.Op("RY(%g)" % (0.2 + 0.1 * i), 1 + i % N) for i in range(12)]
    full = np.diag(np.exp(1j * np.arange(2 ** N)))
    lst = ops + [bt.ifOp("MZ", 2, "X", "H")] + ops + [bt.OpF("phase", full)] + ops + [bt.Op("MZ", 1)]
    for seed in range(6):
        st = bt.zero_state(N, "c128")
        _, outs = bt.apply(st, lst, track_measurements=True, rng=bt.UniformStream(seed))
        a = bt.zero_state(N, "c128")
        r = bt.UniformStream(seed)
        got = []
        for o in lst:
            got += bt.apply(a, o, track_measurements=True, rng=r)[1]
        assert outs == got
        assert np.abs(st.to_numpy() - a.to_numpy()).max() <= 1e-12
