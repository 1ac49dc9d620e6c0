"""The interpreter with a queue that makes room pass by pass (stream = 1, as
the executors run it) against the queue that is emptied, through the host
emulation: the same states, outcomes and draws, in no more passes on
circuits longer than the queue.

Tolerance: both runs apply the same operators in FP64 in orders that differ
by commuting ones; 400 operators of rounding at most, 400 * 2.2e-16 * a
condition of 10 < 1e-12."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from refcirc import random_spec
from test_interp_emu import CSRC, ROCM_INC, ROOT, SRCS, emu, emu_run  # noqa: F401



@pytest.fixture(scope="module")
def emu_stream(tmp_path_factory):
    d = tmp_path_factory.mktemp("emu")
    src = open(SRCS[0]).read()
    init = "ip.init(prog, slots.data(), T, cmin);"
    assert src.count(init) == 1
    (d / "emu.cpp").write_text(src.replace(init, init + " ip.stream = 1;"))
    so = str(d / "libemu_stream.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM_INC,
                    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-o", so, str(d / "emu.cpp")], check=True)
    L = ctypes.CDLL(so)
    L.emu_error.restype = ctypes.c_char_p
    L.emu_set_exec(0)
    return L


@pytest.mark.parametrize("kinds,noise", [(("gate1", "gate2", "ccx"), None),
                                         (("gate1", "gate2"), ("depolarizing", 0.05, "depolarizing", 0.05)),
                                         (("gate1", "gate2", "chan1", "chan2", "kraus"), None),
                                         (("gate1", "gate2", "ccx", "chan1", "meas", "reset", "ifop"),
                                          ("depolarizing", 0.02, "amplitude_damping", 0.1))])
@pytest.mark.parametrize("N,T,cmin", [(9, 4, 1), (10, 6, 2), (8, 8, 0)])
def test_stream_matches_emptied_queue(emu, emu_stream, bt, N, T, cmin, kinds, noise):
    nm = bt.NoiseModel(*noise) if noise else False
    total = [0, 0]
    for seed in range(3):
        spec = random_spec(N, 250, np.random.default_rng(17 * seed + N), kinds=kinds)
        a, oa, sa = emu_run(emu, bt, spec, N, nm, seed=seed, T=T, cmin=cmin)
        b, ob, sb = emu_run(emu_stream, bt, spec, N, nm, seed=seed, T=T, cmin=cmin)
        if sa[2] or sb[2]:
            continue  # a draw within 1e-9 of its boundary
        assert oa == ob and sa[3] == sb[3]
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.allclose(a, b, rtol=0, atol=1e-12, equal_nan=True)
        total[0] += sa[0]
        total[1] += sb[0]
    if kinds[-1] in ("ccx", "gate2") and T < N:
        assert total[1] < total[0], total
