"""Passes whose CNOTs and SWAPs relabel the tile image instead of being
applied: state vectors and density matrices against the oracle, in the host
emulation of the passes and on the device, with one tile (every pass in one
launch: the image is made plain between passes), several, and ragged tile
widths.

Tolerances: those of the circuit executors (complex128 1e-12, complex64 1e-5,
largest entry error)."""
import numpy as np
import pytest

import oracle as O
from refcirc import to_bt, to_ref
from test_interp_emu import emu, emu_run, emu_run_dm  # noqa: F401

TOL = {"c128": 1e-12, "c64": 1e-5}


def permuting_spec(N, nops, seed):
    """Mostly CNOT / SWAP runs between few rotations, so that many stay
    unfused, and some gates that are no such map (CZ, ISWAP, X)."""
    rng = np.random.default_rng(seed)
    spec = [("gate", "H", q, -1, -2, True) for q in range(1, N + 1)]
    for _ in range(nops):
        a, b = [int(x) for x in rng.choice(np.arange(1, N + 1), 2, replace=False)]
        name = ["CNOT", "SWAP", "CNOT", "SWAP", "CNOT", "CZ", "ISWAP", "RXX(0.7)", "1"][rng.integers(9)]
        if name == "1":
            spec.append(("gate", ["RY(0.3)", "T", "X", "SX"][rng.integers(4)], a, -1, -2, True))
        else:
            spec.append(("gate", name, a, b, -2, True))
    return spec


@pytest.fixture
def tiles(bt):
    from bluetangle_jl_amd import _lib
    L = _lib.lib()

    def set_tiles(T):
        for p in (0, 1):
            _lib.check(L.bt_set_tile_bits(p, T))
    yield set_tiles
    set_tiles(0)


@pytest.mark.parametrize("mode,prec", [(1, "c128"), (2, "c64")])
@pytest.mark.parametrize("N,T", [(2, 2), (5, 5), (9, 4), (9, 6), (10, 9)])
def test_emulated_passes(emu, bt, N, T, mode, prec):
    emu.emu_set_exec(mode)
    try:
        for seed in range(3):
            spec = permuting_spec(N, 120, 10 * N + seed)
            s, _, _ = emu_run(emu, bt, spec, N, T=T, cmin=1)
            ref = O.run_sv(N, to_ref(spec), None, O.uniforms(0, 0, 16), tol=1e-9)[0]
            assert np.abs(s - ref).max() < TOL[prec], seed
        if N <= 5:
            nm = ("depolarizing", 0.02, "depolarizing", 0.03)
            spec = permuting_spec(N, 30, N)
            rho = emu_run_dm(emu, bt, spec, N, bt.NoiseModel(*nm), T=max(T, 4))
            ref = O.run_dm(N, to_ref(spec), O.ref_noise(*nm))
            assert np.abs(rho - ref).max() < TOL[prec]
    finally:
        emu.emu_set_exec(0)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N,T", [(2, 0), (4, 3), (9, 6), (12, 0), (12, 8), (14, 0), (15, 11)])
def test_state_vector(bt, tiles, N, T, prec):
    from bluetangle_jl_amd.circuit import Circuit
    from bluetangle_jl_amd.core import StateVector
    tiles(T)
    for seed in range(3):
        spec = permuting_spec(N, 120, 10 * N + seed)
        s = StateVector(N, prec)
        Circuit(to_bt(spec, bt), N, False).run_on(s)
        ref = O.run_sv(N, to_ref(spec), None, O.uniforms(0, 0, 16), tol=1e-9)[0]
        assert np.abs(s.to_numpy() - ref).max() < TOL[prec], seed


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [2, 4, 6, 7])
def test_density_matrix(bt, N, prec):
    from bluetangle_jl_amd.circuit import Circuit
    nm = ("depolarizing", 0.02, "depolarizing", 0.03)
    spec = permuting_spec(N, 40, N) + [("chan", "amplitude_damping", 0.1, q, -1) for q in range(1, N + 1)]
    spec = spec + permuting_spec(N, 20, N + 50)
    rho = bt.zero_rho(N, prec)
    Circuit(to_bt(spec, bt), N, bt.NoiseModel(*nm)).run_dm(rho)
    ref = O.run_dm(N, to_ref(spec), O.ref_noise(*nm))
    assert np.abs(rho.to_numpy() - ref).max() < TOL[prec]
