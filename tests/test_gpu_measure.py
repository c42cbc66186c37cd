"""measure_seq of several qubits in one pass (instruments.hpp:985-1099)
against the oracle: results equal, probabilities and the state left within
1e-12 (a weight is a sum of at most 2^16 products, rounded to 2^-53 each);
complex64 states hold the same inputs exactly and round the result once
(2e-6 with room)."""
import numpy as np
import pytest

from helpers import randket

pytestmark = pytest.mark.gpu


def _targets(n, rng):
    out = [[0], [n - 1], list(range(n)), list(range(n))[::-1]]
    out += [[int(q) for q in rng.permutation(n)[: rng.integers(1, n + 1)]] for _ in range(4)]
    return out


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("destructive", [False, True])
@pytest.mark.parametrize("n", [1, 2, 5, 7, 12, 16])
def test_ket(qa, orc, n, destructive, dtype):
    rng = np.random.default_rng(n)
    dt, tol = (qa.C128, 1e-12) if dtype == "c128" else (qa.C64, 2e-6)
    psi = randket(2 ** n, rng)
    if dtype == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    for t in _targets(n, rng):
        u = float(rng.random())
        st = qa.State.from_array(psi, [2] * n, dtype=dt)
        res, ps = st.measure_seq(t, u, destructive)
        r, p, left = orc.measure_seq(psi, t, 2, destructive, u)
        assert list(r) == res, (t, u)
        assert np.max(np.abs(np.array(ps) - p)) <= tol, (t, u)
        assert np.max(np.abs(st.download().reshape(-1) - np.asarray(left).reshape(-1))) <= tol, (t, u)
        assert st.dims == ([2] * (n - len(t)) or [1] if destructive else [2] * n)


@pytest.mark.parametrize("destructive", [False, True])
@pytest.mark.parametrize("n", [1, 2, 4, 6])
def test_rho(qa, orc, n, destructive):
    rng = np.random.default_rng(n)
    D = 2 ** n
    vs = [randket(D, rng) for _ in range(3)]
    rho = sum(w * np.outer(v, v.conj()) for w, v in zip((0.5, 0.3, 0.2), vs))
    for t in _targets(n, rng):
        u = float(rng.random())
        st = qa.State.from_array(rho, [2] * n)
        res, ps = st.measure_seq(t, u, destructive)
        r, p, left = orc.measure_seq(rho, t, 2, destructive, u)
        assert list(r) == res and np.max(np.abs(np.array(ps) - p)) <= 1e-12, (t, u)
        assert np.max(np.abs(st.download().reshape(-1) - np.asarray(left).reshape(-1))) <= 1e-12, (t, u)


@pytest.mark.parametrize("destructive", [False, True])
@pytest.mark.parametrize("n,dtype", [(4, "c64"), (6, "c64"), (10, "c128"), (11, "c128"), (11, "c64")])
def test_rho_more(qa, orc, n, dtype, destructive):
    """complex64 density matrices, and those of more than 10 subsystems,
    which are projected from the last target down when destructive
    (instruments.hpp:1055-1095): each probability is conditioned on the
    targets before it in that order."""
    rng = np.random.default_rng(100 + n)
    dt, tol = (qa.C128, 1e-12) if dtype == "c128" else (qa.C64, 2e-6)
    D = 2 ** n
    vs = [randket(D, rng) for _ in range(2)]
    rho = sum(w * np.outer(v, v.conj()) for w, v in zip((0.6, 0.4), vs))
    if dtype == "c64":
        rho = rho.astype(np.complex64).astype(np.complex128)
    for t in ([2, 0, n - 1], [n - 1, 1], [1]):
        u = float(rng.random())
        print(f"rho n={n} {dtype} targets {t} destructive={destructive}", flush=True)
        st = qa.State.from_array(rho, [2] * n, dtype=dt)
        res, ps = st.measure_seq(t, u, destructive)
        r, p, left = orc.measure_seq(rho, t, 2, destructive, u)
        assert list(r) == res and np.max(np.abs(np.array(ps) - p)) <= tol, (t, u)
        assert np.max(np.abs(st.download().reshape(-1) - np.asarray(left).reshape(-1))) <= tol, (t, u)


def test_impossible_result(qa):
    """u = 0 selects index 0 also where its probability is 0; dividing by the
    weight 0 leaves no number behind, as target by target."""
    psi = np.array([0, 0, 1, 0], dtype=complex)
    for dest in (False, True):
        st = qa.State.from_array(psi, [2, 2])
        res, ps = st.measure_seq([0, 1], 0.0, dest)
        assert res == [0, 0] and ps[0] == 0 and np.isnan(st.download().view(float)).all()
