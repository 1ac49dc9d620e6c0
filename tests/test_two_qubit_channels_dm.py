"""Two-qubit channels on a density matrix: a product superoperator is applied
as one factor per qubit, any other as a whole (host emulation and GPU)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
X = np.array([[0, 1], [1, 0]], dtype=complex)
Z = np.diag([1.0, -1.0]).astype(complex)
I2 = np.eye(2, dtype=complex)


def channels(bt):
    """(name, Kraus operators): products (equal and unequal factors, one of
    them non-unital) and channels that are no product, one barely so."""
    nm = bt.noise_model
    prod = [np.kron(a, b) for a in nm("amplitude_damping", 0.3) for b in nm("depolarizing", 0.1)]
    corr = [np.sqrt(0.7) * np.kron(I2, I2), np.sqrt(0.3) * np.kron(X, Z)]
    eps = 1e-6
    near = [np.sqrt(1 - eps) * np.kron(I2, I2), np.sqrt(eps) * np.kron(X, X)]
    cx = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]], dtype=complex)
    return {"depolarizing": nm("depolarizing", 0.2, two_qubit=True), "unequal": prod, "correlated": corr,
            "barely": near, "entangling": [cx]}


def circuits(bt, name, seed):
    """Channels on every ordered pair of three of four qubits, alone and after
    a gate on the same pair, between random rotations."""
    rng = np.random.default_rng(seed)
    ks = channels(bt)[name]
    ops, ref = [], []
    for a, b in [(1, 2), (2, 1), (1, 4), (4, 3), (3, 1)]:
        for q in range(1, 5):
            g = "RY(%r)" % float(rng.uniform(0, 6))
            ops.append(bt.Op(g, q))
            ref.append(O.ref_gate(g, q))
        if rng.random() < 0.6:
            ops.append(bt.Op("CNOT", a, b))
            ref.append(O.ref_gate("CNOT", a, b))
        ops.append(bt.OpQC("noise2", ks, a, b))
        ref.append(O.ref_channel_kraus(ks, a, b))
    return ops, ref


NAMES = ["depolarizing", "unequal", "correlated", "barely", "entangling"]


@pytest.fixture(scope="module")
def emu():
    here = os.path.join(ROOT, "tests", "emu")
    out = os.path.join(here, "libbt_emu.so")
    csrc = os.path.join(ROOT, "bluetangle.jl_amd", "csrc")
    inc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
    tmp = "%s.%d.split" % (out, os.getpid())
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I" + inc,
                    "-I" + os.path.join(ROOT, "include"), "-I" + csrc, "-o", tmp, os.path.join(here, "bt_emu.cpp")],
                   check=True)
    L = ctypes.CDLL(tmp)
    os.unlink(tmp)
    L.emu_error.restype = ctypes.c_char_p
    yield L


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("name", NAMES)
def test_lowering_matches_the_oracle(emu, bt, name, mode):
    from bluetangle_jl_amd.circuit import compile_ir
    N = 4
    ops, ref = circuits(bt, name, 5)
    ir = compile_ir(ops, N, False)
    arr, pool = ir.arrays()
    rho = np.zeros(4 ** N, dtype=np.complex128)
    rho[0] = 1
    stats = np.zeros(5, dtype=np.int64)
    emu.emu_set_exec(mode)
    rc = emu.emu_run_dm(N, arr, len(ir.ops), ir.ntop, pool.ctypes.data_as(ctypes.c_void_p),
                        ctypes.c_int64(pool.size // 2), 6, 1, rho.ctypes.data_as(ctypes.c_void_p),
                        stats.ctypes.data_as(ctypes.c_void_p))
    emu.emu_set_exec(0)
    assert rc == 0, emu.emu_error()
    # entries of size <= 1, a few hundred roundings each
    assert np.abs(rho.reshape((2 ** N, 2 ** N), order="F") - O.run_dm(N, ref)).max() <= 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("c64", 1e-5), ("c128", 1e-12)])
@pytest.mark.parametrize("name", NAMES)
def test_gpu_per_op_and_circuit(bt, name, prec, tol):
    from bluetangle_jl_amd.circuit import Circuit
    ops, ref = circuits(bt, name, 6)
    want = O.run_dm(4, ref)
    rho = bt.zero_rho(4, prec)
    bt.apply(rho, ops)
    assert np.abs(rho.to_numpy() - want).max() <= tol
    rho2 = bt.zero_rho(4, prec)
    Circuit(ops, 4).run_dm(rho2)
    assert np.abs(rho2.to_numpy() - want).max() <= tol
