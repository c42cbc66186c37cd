"""Qudit gates, permutations and partial transposes over every gate
dimension that has a kernel of its own and some that have not, mixed
dimensions and dimensions of 1 among them, against the oracle (apply,
applyCTRL, syspermute, ptranspose: operations.hpp).  Gates 1e-12 in
complex128 and 2e-6 in complex64 (at most 49 products a step on amplitudes
below 1); the maps move values (exact), a ket's partial transpose multiplies
two (one rounding each)."""
import numpy as np
import pytest

from helpers import randket

pytestmark = pytest.mark.gpu

DIMS = [[3] * 5, [4, 4, 4], [5, 5, 3], [2, 3, 2, 5, 3], [6, 2, 7], [3, 1, 3, 2], [7, 7, 2], [2, 1, 2, 2], [3] * 8, [25, 16, 9]]


def _haar(d, rng):
    q, r = np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))
    return q * (np.diag(r) / np.abs(np.diag(r)))


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("dims", DIMS, ids=str)
def test_gates(qa, orc, dims, dtype):
    rng = np.random.default_rng(sum(dims))
    dt, tol = (qa.C128, 1e-12) if dtype == "c128" else (qa.C64, 2e-6)
    n, D = len(dims), int(np.prod(dims))
    states = [randket(D, rng)]
    if D <= 128:
        states.append((rng.standard_normal((D, D)) + 1j * rng.standard_normal((D, D))) / D)
    for psi in states:
        for t in [[0], [n - 1], [n // 2]] + [[int(q) for q in rng.permutation(n)[:2]] for _ in range(3)]:
            DA = int(np.prod([dims[q] for q in t]))
            if DA > 64:
                continue
            U = _haar(DA, rng)
            got = qa.State.from_array(psi, dims, dtype=dt).apply(U, t).download()
            assert np.max(np.abs(got - orc.apply(psi, U, t, dims))) <= tol, t
            for d in set(dims):
                c = [q for q in range(n) if dims[q] == d and q not in t]
                for ctrl in ([c[:1], c[:2][::-1]] if len(c) > 1 else [c[:1]] if c else []):
                    sh = [int(x) for x in rng.integers(0, d, len(ctrl))]
                    got = qa.State.from_array(psi, dims, dtype=dt).apply_ctrl(U, ctrl, t, sh).download()
                    assert np.max(np.abs(got - orc.applyCTRL(psi, U, ctrl, t, dims, sh))) <= tol, (t, ctrl, sh)


@pytest.mark.parametrize("dims", DIMS, ids=str)
def test_maps(qa, orc, dims):
    rng = np.random.default_rng(len(dims))
    n, D = len(dims), int(np.prod(dims))
    psi = randket(D, rng)
    st = qa.State.from_array(psi, dims)
    perm = [int(q) for q in rng.permutation(n)]
    assert np.array_equal(st.syspermute(perm).download(), orc.syspermute(psi, perm, dims))
    if D > 300:
        return
    rho = (rng.standard_normal((D, D)) + 1j * rng.standard_normal((D, D))) / D
    sr = qa.State.from_array(rho, dims)
    assert np.array_equal(sr.syspermute(perm).download(), orc.syspermute(rho, perm, dims))
    for t in ([], [0], [n - 1], perm[:2], perm):
        assert np.array_equal(sr.ptranspose(t).download(), orc.ptranspose(rho, t, dims)), t
        assert np.max(np.abs(st.ptranspose(t).download() - orc.ptranspose(psi, t, dims))) <= 1e-15, t


@pytest.mark.parametrize("n", [1, 4, 8, 9, 10])
def test_ket_ptranspose_qubits(qa, orc, n):
    rng = np.random.default_rng(n)
    psi = randket(2 ** n, rng)
    st = qa.State.from_array(psi, [2] * n)
    for t in ([0], [n - 1], [int(q) for q in rng.permutation(n)[: (n + 1) // 2]], list(range(n))):
        assert np.max(np.abs(st.ptranspose(t).download() - orc.ptranspose(psi, t, 2))) <= 1e-15, t
