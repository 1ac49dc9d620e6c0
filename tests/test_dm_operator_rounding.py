"""Operators of density-matrix passes before they are rounded to FP32: the
factors of a product channel and the scales of a pass's superoperators
(host code of bt_circuit.hpp, compiled here)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EPS = 2.0 ** -53
SRC = r"""
#include "bt_circuit.hpp"
extern "C" int split(const double* kraus, int n, double* out) {
  std::vector<std::vector<btc::cd>> K(n, std::vector<btc::cd>(16));
  for (int i = 0; i < n; i++)
    for (int e = 0; e < 16; e++) K[i][e] = btc::cd(kraus[2 * (16 * i + e)], kraus[2 * (16 * i + e) + 1]);
  std::vector<btc::cd> f[2];
  if (!btc::split_superoperator(btc::superoperator(2, K), &f[0], &f[1])) return 0;
  for (int q = 0; q < 2; q++) memcpy(out + 32 * q, f[q].data(), 256);
  return 1;
}
#ifdef SETTLE
extern "C" void settle(int n, int N, const int* bits, const unsigned long long* ctrl, double* m) {
  std::vector<bti::QOp> slots(n);
  bti::Plan plan{};
  plan.nops = n;
  for (int i = 0; i < n; i++) {
    plan.qidx[i] = n - 1 - i;  // slots are in no order
    bti::QOp& q = slots[n - 1 - i];
    q.k = 2;
    q.bits[0] = bits[2 * i];
    q.bits[1] = bits[2 * i + 1];
    q.ctrl = ctrl[i];
    memcpy(q.m, m + 32 * i, 256);
  }
  btc::settle_scales(plan, slots.data(), N);
  for (int i = 0; i < n; i++) memcpy(m + 32 * i, slots[n - 1 - i].m, 256);
}
#endif
"""


def build(tmp_path, flags):
    src, out = str(tmp_path / "h.cpp"), str(tmp_path / "h.so")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "bluetangle.jl_amd", "csrc"), "-o", out, src] + flags, check=True)
    return ctypes.CDLL(out)


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def superop(kraus):
    """sum K (x) conj(K) over [row, column] bits of vec(rho)."""
    return sum(np.kron(K, K.conj()) for K in kraus)


def products(bt):
    nm = bt.noise_model
    return {
        "depolarizing 0.01": (nm("depolarizing", 0.01), nm("depolarizing", 0.01)),
        "depolarizing 0.3": (nm("depolarizing", 0.3), nm("depolarizing", 0.3)),
        "unequal": (nm("amplitude_damping", 0.3), nm("depolarizing", 0.1)),
        "damping first": (nm("phase_damping", 0.2), nm("amplitude_damping", 0.05)),
        "complex": ([bt.gate["H"] @ bt.gate["T"]], nm("bit_flip", 0.25)),
    }


NAMES = ["depolarizing 0.01", "depolarizing 0.3", "unequal", "damping first", "complex"]


@pytest.mark.parametrize("name", NAMES)
def test_factors_of_a_channel_preserve_the_trace(bt, tmp_path, name):
    """Rows 0 and 3 of each factor add up to those of its qubit's channel, (1, 0,
    0, 1) but for the digits of the gate tables, and each factor is that
    channel: entries of size <= 1 from a few roundings each."""
    lib = build(tmp_path, [])
    ka, kb = products(bt)[name]
    both = np.array([np.asarray(np.kron(a, b), dtype=np.complex128).T for a in ka for b in kb])  # column-major
    out = np.zeros((2, 4, 4), dtype=np.complex128)
    assert lib.split(ptr(np.ascontiguousarray(both)), len(both), ptr(out)) == 1
    for got, kraus in zip(out, (ka, kb)):
        f, want = got.T, superop(kraus)  # column-major
        assert np.abs(f[0] + f[3] - (want[0] + want[3])).max() <= 16 * EPS
        assert np.abs(f - want).max() <= 16 * EPS


def held(m, scaled):
    """FP32's `scaled` as a multiple of m, and how far it is from that multiple,
    the trace of a diagonal input counted eight times more."""
    f = scaled.astype(np.complex64).astype(np.complex128)
    c = np.vdot(m, f).real / np.vdot(m, m).real
    d = f - c * m
    t = (d[0, 0] + d[3, 0] + d[0, 3] + d[3, 3]).real
    return c, ((np.abs(d) ** 2).sum() + 8 * t * t) / c ** 2


def test_scales_of_a_pass_multiply_to_one(bt, tmp_path):
    """One-qubit superoperators become multiples of themselves; the multiples that
    FP32 holds, times the last one's, make one.  What FP32 holds as it is,
    operators on two qubits and controlled ones stay as they are."""
    lib = build(tmp_path, ["-DSETTLE"])
    N, rng = 5, np.random.default_rng(4)
    bits, ctrl, mats, free = [], [], [], []

    def add(b, c, m, scaled):
        bits.append(b)
        ctrl.append(c)
        mats.append(np.array(m, dtype=np.complex128))
        free.append(scaled)

    for q in range(N):
        u, _ = np.linalg.qr(rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2)))
        m = superop([K @ u for K in bt.noise_model("amplitude_damping", 0.1)])
        add((q, q + N) if q % 2 else (q + N, q), 0, m, True)
        if q == 1:
            add((2, 2 + N), 0, superop([np.diag([1, 0]), np.array([[0, 1], [0, 0]])]), False)  # a reset: zeros and ones
        if q == 3:
            add((0, 1), 0, m, False)
            add((4, 4 + N), 1, m, False)
    arr = np.array([m.T for m in mats])
    lib.settle(len(mats), N, ptr(np.array(bits, dtype=np.int32)), ptr(np.array(ctrl, dtype=np.uint64)), ptr(arr))
    total, seen, moved = 1.0, 0, False
    for i, (a, b) in enumerate(zip(mats, (m.T for m in arr))):
        if not free[i]:
            assert np.array_equal(a, b)
            continue
        seen += 1
        top = np.unravel_index(np.abs(a.real).argmax(), a.shape)
        c = b.real[top] / a.real[top]
        assert abs(c - 1) <= 2.0 ** -10
        assert np.abs(b - c * a).max() <= 4 * EPS  # entries below 1: a rounding of b, of c and of the product
        moved = moved or c != 1
        kept, off = held(a, b)
        if seen == 1:  # the scale 1 was among those it could take
            assert off <= held(a, a)[1]
        total *= c if seen == N else kept
    assert seen == N and moved
    assert abs(total - 1) <= 64 * EPS  # five multiples, each from sums of 32 terms


def test_one_superoperator_keeps_its_scale(bt, tmp_path):
    lib = build(tmp_path, ["-DSETTLE"])
    m = superop(bt.noise_model("depolarizing", 0.1)).astype(np.complex128)
    arr = np.array([m.T])
    lib.settle(1, 3, ptr(np.array([1, 4], dtype=np.int32)), ptr(np.zeros(1, dtype=np.uint64)), ptr(arr))
    assert np.array_equal(arr[0].T, m)
