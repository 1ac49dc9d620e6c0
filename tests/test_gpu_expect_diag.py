"""Z strings of a state vector (16-byte loads, one workgroup to many) against
FP64 numpy on the same amplitudes.

Tolerance: the weights and their sum are FP64 (2^N terms added in parts of at
most 2^13 by a tree: 1e-12 of the norm); complex64 amplitudes are exact in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("N", [1, 2, 7, 10, 13, 17, 20])
def test_z_strings(bt, N, prec):
    rng = np.random.default_rng(N)
    v = rng.normal(size=2 ** N) + 1j * rng.normal(size=2 ** N)
    s = bt.from_numpy(v / np.linalg.norm(v), prec)
    w = np.abs(s.to_numpy().astype(np.complex128)) ** 2
    idx = np.arange(2 ** N)
    picks = [[q] for q in {1, N}] + ([[1, N], [N - 1, N], list(range(1, N + 1))] if N > 1 else [])
    for qs in picks:
        par = sum((idx >> (N - q)) & 1 for q in qs) & 1
        got = bt.correlation(s, ",".join("Z" * len(qs)), qs)
        assert abs(complex(got) - (w * (1 - 2 * par)).sum()) < 1e-12, qs


def test_non_finite(bt):
    v = np.ones(16, dtype=complex)
    v[5] = np.nan
    assert np.isnan(complex(bt.correlation(bt.from_numpy(v, "c64"), "Z,Z", [1, 4])).real)
