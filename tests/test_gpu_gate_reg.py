"""Dense 2- to 4-qubit gates and density-matrix gates in registers
(qpp::apply, applyCTRL, operations.hpp:72-372, 616-887) with targets and
controls on every side of the lane bits, against the oracle: 1e-12 in
complex128; in complex64 at most 16 products a step, each rounded to 2^-24,
on amplitudes below 1 (2e-6 with room)."""
import numpy as np
import pytest

from helpers import randket

pytestmark = pytest.mark.gpu


def _haar(d, rng):
    q, r = np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))
    return q * (np.diag(r) / np.abs(np.diag(r)))


def _dt(qa, dtype):
    return (qa.C128, 1e-12) if dtype == "c128" else (qa.C64, 2e-6)


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [2, 3, 5, 6, 7, 8, 9, 10, 11, 13, 17])
def test_ket_gates(qa, orc, n, dtype):
    rng = np.random.default_rng(n)
    dt, tol = _dt(qa, dtype)
    psi = randket(2 ** n, rng)
    for k in (2, 3, 4):
        if k > n:
            continue
        sets = [list(range(k)), list(range(n - k, n)), list(range(n - k, n))[::-1]]
        sets += [[int(q) for q in rng.permutation(n)[:k]] for _ in range(4)]
        for t in sets:
            U = _haar(2 ** k, rng)
            st = qa.State.from_array(psi, [2] * n, dtype=dt)
            assert np.max(np.abs(st.apply(U, t).download() - orc.apply(psi, U, t, 2))) <= tol, (k, t)
            rest = [q for q in range(n) if q not in t]
            for nc in (1, 2):
                if nc > len(rest):
                    continue
                for c in (rest[:nc], rest[-nc:]):
                    sh = [int(x) for x in rng.integers(0, 2, nc)]
                    st = qa.State.from_array(psi, [2] * n, dtype=dt)
                    got = st.apply_ctrl(U, c, t, sh).download()
                    assert np.max(np.abs(got - orc.applyCTRL(psi, U, c, t, 2, sh))) <= tol, (k, t, c, sh)


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 8])
def test_rho_gates(qa, orc, n, dtype):
    rng = np.random.default_rng(50 + n)
    dt, tol = _dt(qa, dtype)
    D = 2 ** n
    rho = (rng.standard_normal((D, D)) + 1j * rng.standard_normal((D, D))) / D  # no symmetry to lean on
    for k in (1, 2, 3):
        if k > n:
            continue
        sets = [list(range(k)), list(range(n - k, n))] + [[int(q) for q in rng.permutation(n)[:k]] for _ in range(3)]
        for t in sets:
            U = _haar(2 ** k, rng)
            st = qa.State.from_array(rho, [2] * n, dtype=dt)
            assert np.max(np.abs(st.apply(U, t).download() - orc.apply(rho, U, t, 2))) <= tol, (k, t)
            rest = [q for q in range(n) if q not in t]
            for nc in (1, 2):
                if nc > len(rest):
                    continue
                for c in (rest[:nc], rest[-nc:]):
                    sh = [int(x) for x in rng.integers(0, 2, nc)]
                    st = qa.State.from_array(rho, [2] * n, dtype=dt)
                    got = st.apply_ctrl(U, c, t, sh).download()
                    assert np.max(np.abs(got - orc.applyCTRL(rho, U, c, t, 2, sh))) <= tol, (k, t, c, sh)
        Ks = [_haar(2 ** k, rng) * 0.5 for _ in range(3)]
        if k <= 2:
            st = qa.State.from_array(rho, [2] * n, dtype=dt)
            t = sets[-1]
            assert np.max(np.abs(st.apply_kraus(Ks, t).download() - orc.apply_kraus(rho, Ks, t, 2))) <= tol, t


@pytest.mark.parametrize("n,k,ctrl,dtype", [(11, 1, [0, 1], "c128"), (11, 1, [1, 0, 10], "c128"),
                                            (11, 1, [0, 10], "c128"), (12, 1, [2, 0], "c64"),
                                            (12, 2, [5, 0, 1], "c64"), (12, 2, [0, 11], "c64")])
def test_rho_gates_under_many_controls(qa, orc, n, k, ctrl, dtype):
    """Density matrices large enough that two and more controls above the
    lane bits take rows and columns in a pass each, and neighbours that do
    not."""
    rng = np.random.default_rng(n + len(ctrl))
    dt, tol = _dt(qa, dtype)
    D = 2 ** n
    rho = (rng.standard_normal((D, D)) + 1j * rng.standard_normal((D, D))) / D
    U, t, sh = _haar(2 ** k, rng), [6, 3][:k], [int(x) for x in rng.integers(0, 2, len(ctrl))]
    print(f"rho n={n} k={k} controls {ctrl} {dtype}", flush=True)
    st = qa.State.from_array(rho, [2] * n, dtype=dt)
    got = st.apply_ctrl(U, ctrl, t, sh).download()
    assert np.max(np.abs(got - orc.applyCTRL(rho, U, ctrl, t, 2, sh))) <= tol


@pytest.mark.parametrize("k", [4, 5])
def test_gates_from_two_threads(qa, k):
    """Commuting (diagonal) gates applied to one state by two threads at once,
    each call with a table of its own in device memory: the product of all,
    whatever the order."""
    import threading
    n, reps = 10, 200
    rng = np.random.default_rng(k)
    psi = randket(2 ** n, rng)
    phases = [np.exp(2j * np.pi * rng.random(2 ** k) / reps) for _ in range(2)]
    st = qa.State.from_array(psi, [2] * n)
    t = list(range(2, 2 + k))

    def work(d):
        for _ in range(reps):
            st.apply(np.diag(d), t)

    threads = [threading.Thread(target=work, args=(d,)) for d in phases]
    for x in threads:
        x.start()
    for x in threads:
        x.join()
    want = psi.reshape(4, 2 ** k, -1) * ((phases[0] * phases[1]) ** reps)[None, :, None]
    assert np.max(np.abs(st.download() - want.reshape(-1))) <= 1e-12  # 400 products of modulus 1
