"""The tile pass at the edges of its dispatch: states whose per-thread byte
offsets need 64 bits (2^30 complex64, 2^29 complex128 entries and up), and
every mix of staged operator widths."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,N", [("c64", 29), ("c64", 30), ("c128", 28), ("c128", 29)])
def test_offset_widths(bt, prec, N):
    """Rotations on every qubit and a long-range entangler, then the inverse:
    back to |0...0>; in between, the amplitudes of a product state.  On either
    side of the 32-bit offset limit."""
    from bluetangle_jl_amd.circuit import Circuit
    th = [0.3 + 0.1 * q for q in range(N)]
    rot = [bt.Op("RY(%r)" % th[q - 1], q) for q in range(1, N + 1)]
    ent = [bt.Op("CZ", q, N + 1 - q) for q in range(1, N // 2)]
    inv = [bt.Op("RY(%r)" % -th[q - 1], q) for q in range(1, N + 1)]
    st = bt.zero_state(N, prec)
    Circuit(rot, N, None).run_on(st)
    rng = np.random.default_rng(N)
    idx = rng.integers(0, 1 << N, 64, dtype=np.uint64)
    want = np.array([np.prod([np.sin(t / 2) if (int(i) >> (N - 1 - q)) & 1 else np.cos(t / 2)
                              for q, t in enumerate(th)]) for i in idx])
    # one rounding per operator and amplitude: N of them, of a product of at most 1
    tol = N * (2.0 ** -23 if prec == "c64" else 2.0 ** -52)
    assert np.abs(st.gather(idx) - want).max() <= tol
    Circuit(ent + ent + inv, N, None).run_on(st)
    a = st.gather([0, 1, 1 << (N - 1)])
    assert abs(a[0] - 1) <= 4 * tol and np.abs(a[1:]).max() <= 4 * tol
    assert abs(st.norm2() - 1) <= 8 * tol


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [6, 13, 15])
def test_staged_operator_widths(bt, prec, N):
    """One-, two-, three- and four-bit operators (in-tile controls widen a
    gate) in the same passes, against the oracle."""
    from bluetangle_jl_amd.circuit import Circuit
    rng = np.random.default_rng(77 + N)
    ops_bt, ops_ref = [], []

    def haar(d):
        q, r = np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))
        return q * (np.diag(r) / np.abs(np.diag(r)))

    for i in range(40):
        a, b, c = (int(x) + 1 for x in rng.permutation(N)[:3])
        kind = i % 4
        if kind == 0:
            u = haar(2)
            ops_bt.append(bt.Op("U1", u, a))
            ops_ref.append(O.ref_gate("U1", a, mat=u))
        elif kind == 1:
            u = haar(4)
            ops_bt.append(bt.Op("U2", u, a, b))
            ops_ref.append(O.ref_gate("U2", a, b, mat=u))
        elif kind == 2:
            u = haar(2)
            ops_bt.append(bt.Op("UC", u, a, control=b))
            ops_ref.append(O.ref_gate("UC", a, control=b, mat=u))
        else:
            m = bt.gate["CX"]
            ops_bt.append(bt.Op("CX", m, a, b, control=c))
            ops_ref.append(O.ref_gate("CX", a, b, control=c, mat=m))
    r = O.run_sv(N, ops_ref, None, O.uniforms(0, 0, 16))[0]
    st = bt.zero_state(N, prec)
    Circuit(ops_bt, N, None).run_on(st)
    # 40 operators of at most 16 products per amplitude
    assert np.abs(st.to_numpy() - r).max() <= 40 * 16 * (2.0 ** -24 if prec == "c64" else 2.0 ** -53)
