"""Shots of sparse states at the boundaries of their cumulative sums: an index
next to the boundary, never one without probability."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _noalloc(bt, st, u):
    L = bt.core.L
    out, nb = np.zeros(len(u), dtype=np.uint64), ctypes.c_int64()
    L.check(L.lib().bt_sample_noalloc(st.handle, len(u), L.dptr(u), out.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64)),
                                      ctypes.byref(nb)))
    return out.astype(np.int64), nb.value


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [13, 16, 18, 20, 22, 23])
def test_boundaries_between_distant_chunks(bt, N, prec):
    """K equal amplitudes in chunks of their own, u = j / K: entry j - 1 or j."""
    rng = np.random.default_rng(N)
    chunks = 2 ** N // 2048
    st = bt.zero_state(N, prec)
    for K in (3, 5, 7, 11, 13, 24, 31):
        if K > chunks:
            continue
        for _ in range(4):
            at = np.sort(rng.choice(chunks, K, replace=False)) * 2048 + rng.integers(0, 2048, K)
            v = np.zeros(2 ** N, dtype=np.complex128)
            v[at] = 1 / np.sqrt(K)
            st.upload(v)
            u = np.arange(K) / K
            for got, flagged in (bt.measurement.sample_with(st, u), _noalloc(bt, st, u)):
                which = np.searchsorted(at, got)
                assert np.array_equal(at[np.minimum(which, K - 1)], got)  # an entry with probability
                j = np.arange(K)
                assert np.all((which == j) | (which == j - 1))
                assert flagged == K  # every target lies on a boundary


@pytest.mark.parametrize("N,at", [(12, [4095]), (18, [2 ** 17 + 5]), (23, [0, 2 ** 22, 2 ** 23 - 1])])
def test_probability_at_the_ends(bt, N, at):
    """The last chunks, or all but one, hold nothing: the largest uniform still finds an entry."""
    v = np.zeros(2 ** N, dtype=np.complex128)
    v[at] = 0.3
    st = bt.from_numpy(v, "c128")
    got, _ = bt.measurement.sample_with(st, np.array([0.0, 0.5, 1 - 2.0 ** -53]))
    assert got[0] == at[0] and got[2] == at[-1] and got[1] in at
