"""The tuning that is reported and chosen is the one noisy trajectories run at."""
import ctypes

import numpy as np
import pytest

from refcirc import brickwork_spec, to_bt


def _tuning(prec):
    from bluetangle_jl_amd import _lib as L
    got = [ctypes.c_int() for _ in range(3)]
    L.check(L.lib().bt_get_tuning(prec, *[ctypes.byref(g) for g in got]))
    return [g.value for g in got]


@pytest.mark.parametrize("prec,bits", [(0, 3), (1, 2)])
def test_reported_default(bt, prec, bits):
    """Circuits that decide branches keep one bit fewer than full passes."""
    from bluetangle_jl_amd import _lib as L
    L.check(L.lib().bt_set_tuning(prec, 0, 0, 0))
    assert _tuning(prec)[1] == bits
    L.check(L.lib().bt_set_tuning(prec, 0, 5, 0))
    try:
        assert _tuning(prec)[1] == 5
    finally:
        L.check(L.lib().bt_set_tuning(prec, 0, 0, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("prec,name,bits", [(0, "c64", 3), (1, "c128", 2)])
def test_a_default_that_wins_stays_a_default(bt, prec, name, bits):
    """The default is among the candidates; where it wins, gate-only circuits
    still plan by their own rule, where another wins, by what was set."""
    from bluetangle_jl_amd import _lib as L
    from bluetangle_jl_amd.circuit import Circuit
    N = 15
    noise = bt.NoiseModel("depolarizing", 1e-3, "depolarizing", 1e-2)
    noisy = Circuit(to_bt(brickwork_spec(N, 3, 4, ad_gamma=5e-3, mz_prob=0.2), bt), N, noise)
    gates = to_bt(brickwork_spec(N, 12, 5), bt)

    def passes():
        return Circuit(gates, N).run_on(bt.zero_state(N, name))[1]["passes"]

    by_rule = passes()
    try:
        t = noisy.autotune(name, sample=8)
        assert t["coalesce_bits"] in {bits, 3, 4, 5}
        assert _tuning(prec) == [t["tile_bits"], t["coalesce_bits"], t["tiles_per_block"]]
        tuned = passes()
        L.check(L.lib().bt_set_tuning(prec, t["tile_bits"], 0 if t["coalesce_bits"] == bits else t["coalesce_bits"], 0))
        assert tuned == passes()
        L.check(L.lib().bt_set_tuning(prec, 0, 0, 0))
        assert passes() == by_rule
    finally:
        L.check(L.lib().bt_set_tuning(prec, 0, 0, 0))
