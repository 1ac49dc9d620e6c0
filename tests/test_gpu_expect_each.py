"""<P_b> of every qubit in a few reads of the state (bt_expect_each), and the
reductions whose last workgroup adds the totals, at the edges of their tiles
and launch sizes, against numpy in FP64."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(bt, N, prec, seed):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=2 ** N) + 1j * rng.normal(size=2 ** N)
    v[rng.integers(0, 2 ** N, max(1, 2 ** N // 8))] = 0
    v /= np.linalg.norm(v) * 0.7  # not normalised
    if prec == "c64":
        v = v.astype(np.complex64).astype(np.complex128)
    return bt.from_numpy(v, prec), v


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [1, 2, 4, 5, 11, 12, 13, 15, 19, 20, 21])
def test_every_qubit(bt, N, prec):
    st, v = _state(bt, N, prec, 100 + N)
    n2 = float(np.sum(np.abs(v) ** 2))
    for name in "XYZ":
        got = bt.expect(st, name)
        want = []
        for q in range(1, N + 1):
            w = v.reshape(2 ** (q - 1), 2, -1)
            a, b = w[:, 0, :], w[:, 1, :]
            z = np.vdot(a, b)
            want.append(2 * z.real if name == "X" else 2 * z.imag if name == "Y" else
                        float(np.sum(np.abs(a) ** 2) - np.sum(np.abs(b) ** 2)))
        # FP64 sums of 2^N terms that add up to at most n2 in size
        assert np.abs(got - np.array(want)).max() <= 2.0 ** -50 * max(N, 4) * n2 * 8
        # the same as one qubit at a time
        one = np.array([bt.expect(st, name, q) for q in range(1, N + 1)])
        assert np.abs(got - one).max() <= 2.0 ** -50 * max(N, 4) * n2 * 8


def test_every_qubit_arguments(bt):
    from bluetangle_jl_amd import _lib
    out = np.zeros(4)
    rho = bt.zero_rho(2, "c64")
    assert _lib.lib().bt_expect_each(rho.handle, 3, _lib.dptr(out)) == -2
    st = bt.zero_state(3, "c64")
    for bad in (0, 4, -1):
        assert _lib.lib().bt_expect_each(st.handle, bad, _lib.dptr(out)) == -1
    assert _lib.lib().bt_expect_each(st.handle, 3, None) == -1


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [3, 8, 9, 18, 20])
def test_reductions_add_up_whatever_the_launch(bt, N, prec):
    """Reduced rho over 1 to 3 bits, the norm and an inner product: one
    workgroup, a few, and the most (2^20 amplitudes); twice in a row, the
    second time bit for bit the same."""
    from bluetangle_jl_amd import _lib
    st, v = _state(bt, N, prec, 7 * N)
    n2 = float(np.sum(np.abs(v) ** 2))
    tol = 2.0 ** -50 * N * n2 * 8
    assert st.norm2() == st.norm2() and abs(st.norm2() - n2) <= tol
    other = st.copy()
    assert abs(st.inner(other) - n2) <= tol and st.inner(other) == st.inner(other)
    for bits in ([0], [N - 1], [1, 0], [N - 1, 0], [2, 0, 1], [N - 1, 1, 0]):
        k = len(bits)
        out = []
        for _ in range(2):
            rho, t = np.zeros(2 * 4 ** k), ctypes.c_double()
            b = np.array(bits, dtype=np.int32)
            _lib.check(_lib.lib().bt_reduced_rho(st.handle, k, _lib.iptr(b), _lib.dptr(rho), ctypes.byref(t)))
            out.append(rho)
            assert abs(t.value - n2) <= tol
        assert np.array_equal(out[0], out[1])
        w = np.moveaxis(v.reshape([2] * N), [N - 1 - x for x in bits], range(k)).reshape(2 ** k, -1)
        want = w @ w.conj().T
        assert np.abs(out[0].view(np.complex128).reshape(2 ** k, 2 ** k, order="F") - want).max() <= tol
