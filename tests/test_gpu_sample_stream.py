"""Shot sampling at the edges of its rows, chunks and scan runs, and shots on
the counter stream against the same uniforms passed in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [1, 2, 5, 6, 7, 10, 11, 12, 14, 22, 23])
def test_rule_and_stream(bt, N, prec):
    """Smallest i with u T < C_i on a state with runs of exact zeros; 2^22 and
    2^23 amplitudes have one and two runs of the scan (2048 chunks each)."""
    rng = np.random.default_rng(50 + N)
    v = (rng.normal(size=2 ** N) + 1j * rng.normal(size=2 ** N)).astype(np.complex64).astype(np.complex128)
    v[rng.random(2 ** N) < 0.3] = 0
    if N >= 11:
        v[100:2200] = 0  # more than a whole chunk
        v[-700:] = 0
    v[2 ** N // 3] = 0.5
    st = bt.from_numpy(v, prec)
    shots = 3000
    u = np.array([bt._lib.lib().bt_uniform(9, 4, 17 + i) for i in range(shots)])
    got, nb = bt.measurement.sample_with(st, u)
    c = np.cumsum(np.abs(v) ** 2)
    want = np.searchsorted(c, u * c[-1], side="right")
    # FP64 sums of 2^N terms in another order: off by less than this of the total
    near = np.abs(np.take(c, want) - u * c[-1]) <= 1e-12 * c[-1]
    near |= np.abs(np.where(want > 0, np.take(c, want - 1), 0.0) - u * c[-1]) <= 1e-12 * c[-1]
    assert np.array_equal(got[~near], want[~near])
    assert np.all(np.abs(v[got]) > 0)
    assert nb <= near.sum() + 1
    rs = bt.UniformStream(9, 4)
    rs.draw = 17
    assert np.array_equal(bt.sample(st, shots, rs), got) and rs.draw == 17 + shots
    # another callable draws for itself
    it = iter(u)
    assert np.array_equal(bt.sample(st, shots, lambda: next(it)), got)
    # fewer and more shots than the kept buffers hold
    assert np.array_equal(bt.measurement.sample_with(st, u[:1])[0], got[:1])
    assert np.array_equal(bt.measurement.sample_with(st, u)[0], got)


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_degenerate_states(bt, prec):
    st = bt.zero_state(5, prec)
    assert np.all(bt.sample(st, 7, bt.UniformStream(1)) == 0)
    st.upload(np.zeros(32))
    assert np.all(bt.sample(st, 7, bt.UniformStream(1)) == 0)
    assert bt.measurement.sample_with(st, [0.25])[1] == 1  # flagged
    assert bt.sample(st, 0, bt.UniformStream(1)).size == 0
    with pytest.raises(TypeError):
        bt.sample(bt.zero_rho(2, prec), 3)
