"""Errors of a run of operations (bt_apply_ops): which of them send the list
through the per-op entries, and that none is applied twice."""
import ctypes

import numpy as np
import pytest


class _Entries:
    """A library whose entries for runs of operations answer `code`."""

    def __init__(self, code):
        self.code, self.calls = code, 0

    def __getattr__(self, name):
        assert name.startswith("bt_apply_ops")
        return self._answer

    def _answer(self, *args):
        self.calls += 1
        return self.code

    def bt_last_error(self):
        return b"planted"


@pytest.mark.parametrize("code", [-3, -6])
def test_an_error_after_passes_is_raised(bt, monkeypatch, code):
    """BT_ERR_HIP and BT_ERR_STATE may come from the middle of a run: the list
    is not applied again op by op."""
    from bluetangle_jl_amd import core
    st = core.StateVector.__new__(core.StateVector)
    st.handle, st.N, st.prec = None, 3, 1
    fake = _Entries(code)
    monkeypatch.setattr(core.L, "lib", lambda: fake)
    monkeypatch.setattr(core, "_apply_one", lambda *a: pytest.fail("applied a second time"))
    ops = [bt.Op("H", 1 + i % 3) for i in range(10)] + [bt.Op("MZ", 1)]
    with pytest.raises(RuntimeError):
        core._apply_run(st, ops, False, None, iter(np.linspace(0.1, 0.9, 9)).__next__, [])
    assert fake.calls == 1


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("value", [0.0, float("nan"), float("inf")])
def test_no_norm_has_a_code_of_its_own(bt, prec, value):
    from bluetangle_jl_amd.circuit import compile_ir
    L = bt.core.L
    st = bt.zero_state(3, prec)
    st.upload(np.full(8, value, dtype=np.complex128))
    before = st.to_numpy()
    ir = compile_ir([bt.Op("H", 1), bt.Op("MZ", 1)], 3)
    arr, pool = ir.arrays()
    u, out, n = np.array([0.3]), np.zeros(4, dtype=np.int32), ctypes.c_int64()
    rc = L.lib().bt_apply_ops(st.handle, arr, 2, L.dptr(pool), pool.size // 2, L.dptr(u), 1, L.iptr(out), 4,
                              ctypes.byref(n))
    assert rc == -9 and n.value == 0
    assert np.array_equal(before, st.to_numpy(), equal_nan=True)
