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


class _Counted:
    """A caller's own rng: the counter stream's draws, `most` of them."""

    def __init__(self, bt, seed, most=10 ** 9):
        self.stream, self.given, self.most = bt.UniformStream(seed), 0, most

    def __call__(self):
        if self.given == self.most:
            raise StopIteration("no more draws")
        self.given += 1
        return self.stream()


def _both_ways(bt, N, ops, prec, seed, most=10 ** 9):
    """(error type, outcomes, draws, state) of the list and of its operations one by one."""
    res = []
    for one in (False, True):
        st = bt.zero_state(N, prec)
        rng, outs, err = _Counted(bt, seed, most), [], None
        try:
            if one:
                for o in ops:
                    outs += bt.apply(st, o, track_measurements=True, rng=rng)[1]
            else:
                outs = bt.apply(st, ops, track_measurements=True, rng=rng)[1]
        except Exception as e:
            err, outs = type(e), None
        res.append((err, outs if err is None else None, rng.given, st.to_numpy()))
    return res


def _spread(bt, N):
    return [bt.Op("RY(%g)" % (0.3 + 0.2 * i), 1 + i % N) for i in range(11)]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_channel_of_many_kraus_operators(bt, prec):
    """65 Kraus operators are more than a circuit takes; the list goes op by op, on the same draws."""
    N = 5
    many = [np.eye(2) / np.sqrt(65)] * 65
    ops = _spread(bt, N) + [bt.Op("MZ", 2), bt.OpQC("many", many, 3), bt.OpQC("amplitude_damping", 0.3, 1), bt.Op("MX", 3)]
    for seed in range(4):
        a, b = _both_ways(bt, N, ops, prec, seed)
        assert a[:3] == b[:3] and a[0] is None and np.array_equal(a[3], b[3])


@pytest.mark.gpu
def test_operation_wider_than_the_tile(bt):
    """Three-qubit channels under tiles of two bits: op by op, not half a run."""
    N, L = 5, bt.core.L
    k3 = [np.sqrt(0.9) * np.eye(8), np.sqrt(0.1) * np.kron(np.kron(bt.gate["X"], bt.gate["Z"]), bt.gate["Y"])]
    ops = _spread(bt, N) + [bt.Op("MZ", 1), bt.OpQC("three", k3, 2), bt.Op("MZ", 4)]
    L.check(L.lib().bt_set_tile_bits(1, 2))
    try:
        a, b = _both_ways(bt, N, ops, "c128", 3)
    finally:
        L.check(L.lib().bt_set_tile_bits(1, 0))
    assert a[:3] == b[:3] and a[0] is None and np.array_equal(a[3], b[3])


@pytest.mark.gpu
@pytest.mark.parametrize("most", [0, 1, 3])
def test_rng_that_gives_out(bt, most):
    """The operations before the draw that cannot be had are applied, and the rng's error is raised."""
    N = 4
    ops = _spread(bt, N) + [bt.OpQC("amplitude_damping", 0.2, 1), bt.Op("MZ", 2), bt.Op("H", 3), bt.OpQC("phase_damping", 0.3, 2),
                            bt.Op("MY", 4)]
    a, b = _both_ways(bt, N, ops, "c128", 1, most)
    assert a[:3] == b[:3] and a[0] is StopIteration and np.array_equal(a[3], b[3])


@pytest.mark.gpu
@pytest.mark.parametrize("bad", ["qubit", "name", "model"])
def test_draws_before_an_error(bt, bad):
    """A list that raises at an operation has drawn for the ones before it only."""
    N = 4
    ops = _spread(bt, N) + [bt.Op("MZ", 2), bt.OpQC("amplitude_damping", 0.2, 1), bt.Op("H", 1)]
    wrong = {"qubit": bt.Op("CNOT", 1, 9), "name": bt.Op("MZ", 3), "model": bt.OpQC("amplitude_damping", 0.1, 9)}[bad]
    if bad == "name":
        wrong.name = "MQ"
    a, b = _both_ways(bt, N, ops + [wrong] + ops, "c128", 2)
    assert a[:3] == b[:3] and a[0] is not None and a[2] == 2
    assert np.abs(a[3] - b[3]).max() <= 1e-13


def test_long_lists_are_several_runs(bt, monkeypatch):
    """A run holds the tables of all its passes, so a list of any length is taken in pieces."""
    from bluetangle_jl_amd import core
    st = core.StateVector.__new__(core.StateVector)
    st.N, st.prec, st.handle = 3, 1, None
    seen = []
    monkeypatch.setattr(core, "_apply_run", lambda state, run, *a: seen.extend([len(run)]) or True)
    monkeypatch.setattr(core, "_apply_one", lambda state, op, *a: seen.append(op.name))
    core._apply_list(st, [bt.Op("H", 1)] * 10000 + [bt.ifOp("MZ", 2, "X", "H")] + [bt.Op("H", 1)] * 4097, False, False,
                     None, None, [])
    assert seen == [4096, 4096, 1808, "MZ", 4096, "H"]


def test_measurements_do_not_make_a_run(bt, monkeypatch):
    """Short lists with measurements or resets are as fast op by op; gates and channels alone make a run of ten."""
    from bluetangle_jl_amd import core
    seen = []
    monkeypatch.setattr(core, "_apply_run", lambda state, run, *a: seen.append(len(run)) or True)
    monkeypatch.setattr(core, "_apply_one", lambda state, op, *a: seen.append(op.name))

    def routes(N, ops):
        st = core.StateVector.__new__(core.StateVector)
        st.N, st.prec, st.handle = N, 0, None
        seen.clear()
        core._apply_list(st, ops, False, False, None, None, [])
        return list(seen)

    h, mz, res, damp = bt.Op("H", 1), bt.Op("MZ", 1), bt.Op("RES", 2), bt.OpQC("amplitude_damping", 0.1, 1)
    assert routes(12, [h] * 10) == [10] and routes(12, [h] * 9) == ["H"] * 9
    assert routes(12, [h] * 5 + [damp] * 5) == [10]
    assert routes(12, [h] * 15 + [mz]) == ["H"] * 15 + ["MZ"] and routes(12, [h] * 16 + [mz] * 3) == [19]
    assert routes(12, [res] + [h] * 15)[1:] == ["H"] * 15 and routes(12, [res] + [h] * 16) == [17]
    assert routes(23, [h] * 4) == [4] and routes(23, [h] * 3) == ["H"] * 3
    assert routes(23, [h] * 9 + [mz]) == ["H"] * 9 + ["MZ"] and routes(23, [h] * 10 + [mz]) == [11]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_list_on_a_state_without_a_norm(bt, prec):
    """A list long enough for a run, on a zero state: op by op, on the same draws."""
    ops = [bt.Op("H", 1 + i % 3) for i in range(20)] + [bt.Op("MZ", 1), bt.Op("MR", 2), bt.OpQC("depolarizing", 0.1, 3)]
    res = []
    for one in (False, True):
        st, rng, outs = bt.zero_state(3, prec), _Counted(bt, 3), []
        st.upload(np.zeros(8))
        if one:
            for o in ops:
                outs += bt.apply(st, o, track_measurements=True, rng=rng)[1]
        else:
            outs = bt.apply(st, ops, track_measurements=True, rng=rng)[1]
        res.append((outs, rng.given, st.to_numpy()))
    assert res[0][:2] == res[1][:2] and np.array_equal(res[0][2], res[1][2], equal_nan=True)
