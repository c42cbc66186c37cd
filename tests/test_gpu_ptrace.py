"""Partial traces at the edges of the kernels' tiles and splits, against the
oracle (qpp::ptrace, operations.hpp:1908-2114).

A partial trace entry is a sum of Dsub products of amplitudes of a unit
state; in FP64 its error is below Dsub * 2^-53 times the sum of their
moduli (at most 1), and complex64 adds one rounding of the result and the
inputs are exact in both, so 1e-13 and 1e-6 hold with room at these sizes."""
import numpy as np
import pytest

from helpers import randket

pytestmark = pytest.mark.gpu

QUBITS = [
    # (n, traced): kept 1..16 states (rows filled with traced digits), tiles of
    # 32 rows with and without a remainder slice, all or nothing traced
    (16, list(range(1, 16))), (16, list(range(15))), (17, [0, 2, 3, 4, 6, 7, 8, 9, 11, 12, 13, 14, 16]),
    (14, list(range(4, 14))), (14, list(range(10))), (15, [1, 3, 5, 7, 9, 11, 13]), (13, [0, 1, 2, 12]),
    (12, list(range(12))), (10, []), (12, [3, 4]), (6, [0, 5]), (18, [17, 0, 4, 5, 9, 10, 11, 12, 13, 14, 15, 16]),
]
QUDITS = [
    ([3] * 10, [0, 1, 2, 4, 5, 6, 7, 9]), ([3] * 9, [1, 2, 3, 8]), ([5] * 7, [0, 2, 3, 4, 5, 6]),
    ([4, 3, 2, 5, 3, 7, 2], [1, 3, 4, 5]), ([2, 1, 300, 16, 3], [2]), ([2, 33, 1, 40, 5], [3, 1]), ([7, 2500, 3], [1]), ([5000, 13], [0]),
    ([6, 11, 13, 17], [3, 0]),
]


# large enough for the matrix products: rows at the edges of their tiles (16,
# 32, 64 and one more), traced digits inside a slice's step and across slices,
# rows along and across the fastest digit; and shapes on either side of the
# rule that chooses them
PRODUCTS = [
    ([16] + [2] * 13, list(range(1, 14))), ([2] * 13 + [16], list(range(13))), ([17, 2, 4, 8, 4, 8, 4], [1, 2, 3, 4, 5, 6]),
    ([32] + [2] * 13, list(range(1, 14))), ([2] * 12 + [33], list(range(12))), ([8, 3, 8, 5, 8, 3, 9], [1, 3, 4, 5, 6]),
    ([64] + [2] * 11, list(range(1, 12))), ([2] * 11 + [65], list(range(11))), ([3] * 11, [0, 1, 3, 5, 7, 10]),
    ([129, 5, 3, 7, 4], [1, 2, 3, 4]), ([4, 31, 9, 31], [0, 2]), ([81, 1000], [1]), ([1000, 30], [0]), ([17, 4000], [1]),
    ([3] * 9, [4, 5, 6, 7, 8]), ([50, 20, 100], [1, 2]), ([40, 4096], [1]), ([300, 4096], [1]),
    ([500, 600], [0]),
]


def _check(qa, orc, dims, traced, dtype, rng):
    psi = randket(int(np.prod(dims)), rng)
    if dtype == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    st = qa.State.from_array(psi, dims, dtype=qa.C128 if dtype == "c128" else qa.C64)
    got = st.ptrace(traced).download().astype(np.complex128)
    assert np.max(np.abs(got - orc.ptrace(psi, traced, dims))) <= (1e-13 if dtype == "c128" else 1e-6)
    return got


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n,traced", QUBITS)
def test_ptrace_ket_qubits(qa, orc, n, traced, dtype):
    got = _check(qa, orc, [2] * n, traced, dtype, np.random.default_rng(n + len(traced)))
    if 2 * n - len(traced) >= 16 and len(traced) >= 4:  # the matrix products: one triangle mirrored
        assert np.array_equal(got, got.conj().T)


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("dims,traced", QUDITS)
def test_ptrace_ket_qudits(qa, orc, dims, traced, dtype):
    _check(qa, orc, dims, traced, dtype, np.random.default_rng(len(dims)))


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("dims,traced", PRODUCTS)
def test_ptrace_ket_products(qa, orc, dims, traced, dtype):
    got = _check(qa, orc, dims, traced, dtype, np.random.default_rng(len(dims) + dims[0]))
    assert np.array_equal(got, got.conj().T)  # either way one triangle is the other's conjugate


@pytest.mark.parametrize("dims,traced", [([2] * 9, [0]), ([2] * 9, [8]), ([2] * 9, list(range(1, 9))), ([2] * 9, [2, 5, 0]),
                                         ([3] * 5, [1, 4]), ([3, 2, 1, 5, 4], [3, 0]), ([500], [0]), ([7, 60], [1])])
def test_ptrace_rho(qa, orc, dims, traced):
    rng = np.random.default_rng(11)
    D = int(np.prod(dims))
    rho = (rng.standard_normal((D, D)) + 1j * rng.standard_normal((D, D))) / D
    for dtype, tol in ((qa.C128, 1e-13), (qa.C64, 1e-6)):
        got = qa.State.from_array(rho, dims, dtype=dtype).ptrace(traced).download()
        assert np.max(np.abs(got - orc.ptrace(rho, traced, dims))) <= tol
