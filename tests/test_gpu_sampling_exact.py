"""The exact sampling table on the device (every shot forced through it)
against the oracle's libstdc++ restatement, including uniforms on and next to
the cumulative table's edges, zero runs, one dominant weight, amplitudes
spanning hundreds of binades and exact powers of two, up to 22 qubits."""
import numpy as np
import pytest

from helpers import randket

pytestmark = pytest.mark.gpu


def make_state(mode, n, rng):
    D = 2 ** n
    if mode == "random":
        psi = randket(D, rng)
        if n >= 9:
            psi[rng.integers(D, size=D // 4)] = 0
    elif mode == "dominant":
        psi = randket(D, rng) * 1e-9
        psi[D // 3] = np.sqrt(0.75)
    elif mode == "tiny":  # |a| from 1e-150 to 1: p across ~1000 binades
        psi = 10.0 ** (-150.0 * rng.random(D)) * np.exp(2j * np.pi * rng.random(D))
        psi[0] = 1e-160
    elif mode == "powers":  # p = 2^-k exactly (left unnormalised: the
        # table divides by the sum)
        return np.ldexp(1.0, -rng.integers(5, 20, size=D)).astype(complex)
    else:
        raise ValueError(mode)
    return psi / np.linalg.norm(psi)


def uniforms(cp, rng, nedge=20):
    u = list(rng.random(200))
    for k in rng.integers(0, len(cp), size=nedge):
        c = float(cp[k])
        u += [c, np.nextafter(c, 0), np.nextafter(c, 1)]
    return [min(x, np.nextafter(1.0, 0)) for x in u] + [np.nextafter(1.0, 0), 1e-300, 0.0]


CASES = [("random", n) for n in (2, 9, 14, 17, 20, 22)] + \
        [(m, n) for m in ("dominant", "tiny", "powers") for n in (12, 20)]


@pytest.mark.parametrize("mode,n", CASES)
def test_forced_exact_table_matches_oracle(qa, orc, mode, n, monkeypatch):
    print(f"exact table: mode={mode} n={n}", flush=True)
    monkeypatch.setenv("QPP_AMD_FORCE_EXACT", "1")
    rng = np.random.default_rng(77 + n)
    psi = make_state(mode, n, rng)
    p = orc.probs(psi)
    cp = orc.discrete_table(p)
    u = uniforms(cp, rng)
    st = qa.State.from_array(psi, [2] * n)
    idx, dig, pr = st.sample(list(range(n)), u)
    # lower_bound in the oracle's sequential table (cp is non-decreasing)
    ref = [int(np.searchsorted(cp, x, side="left")) for x in u]
    assert [int(i) for i in idx] == ref
    if n <= 14:  # the oracle's own draw routine agrees with the table
        assert ref == [orc.discrete_draw(p, x) for x in u]
    assert np.array_equal(pr, p[ref])
    # and the same as the error-bounded parallel search
    monkeypatch.delenv("QPP_AMD_FORCE_EXACT")
    idx2, _, _ = st.sample(list(range(n)), u)
    assert np.array_equal(idx, idx2)


@pytest.mark.parametrize("forced,n,nshots", [(False, 10, 262144), (False, 10, 300001), (True, 10, 300001),
                                             (False, 3, 2 ** 24 + 777), (True, 3, 2 ** 24 + 777)])
def test_more_shots_than_one_launch_of_waves(qa, orc, forced, n, nshots, monkeypatch):
    """More shots than the searches' grids hold at one a wave (262144) or one
    a thread (2^24): every shot is searched and equals the oracle's table."""
    print(f"many shots: forced={forced} n={n} shots={nshots}", flush=True)
    rng = np.random.default_rng(n)
    # another call first, whose workspace the pool may hand out again
    qa.State.from_array(randket(2 ** 9, rng), [2] * 9).sample([0], rng.random(1000))
    if forced:
        monkeypatch.setenv("QPP_AMD_FORCE_EXACT", "1")
    psi = randket(2 ** n, rng)
    p = orc.probs(psi)
    u = rng.random(nshots)
    idx, _, pr = qa.State.from_array(psi, [2] * n).sample([0], u)
    ref = np.searchsorted(orc.discrete_table(p), u, side="left")
    assert np.array_equal(idx, ref.astype(np.uint64))
    assert np.array_equal(pr, p[ref])


@pytest.mark.parametrize("kind,n,nshots", [
    ("ket", 3, 4096), ("ket", 3, 4097), ("ket", 12, 4096), ("ket", 12, 4097), ("ket", 12, 20000), ("ket", 13, 4098),
    ("ket", 14, 4099), ("ket", 14, 4100), ("ket", 20, 4288), ("ket", 20, 4289), ("ket", 20, 255), ("ket", 20, 256),
    ("c64", 13, 3000), ("c64", 13, 9000), ("rho", 5, 4097), ("rho", 7, 100), ("rho", 7, 6000)])
def test_exact_table_by_number_of_shots(qa, orc, kind, n, nshots, monkeypatch):
    """The exact table's three ways (a workgroup per shot, per block, the
    whole table) at the shot counts where one takes over from another: equal
    to the oracle's table, with the probabilities of the state."""
    monkeypatch.setenv("QPP_AMD_FORCE_EXACT", "1")
    rng = np.random.default_rng(n + nshots)
    psi = randket(2 ** n, rng)
    if kind == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    A = np.outer(psi, psi.conj()) if kind == "rho" else psi
    p = orc.probs(A)
    u = np.concatenate([[0.0, np.nextafter(1.0, 0)], rng.random(nshots - 2)])
    st = qa.State.from_array(A, [2] * n, dtype=qa.C64 if kind == "c64" else qa.C128)
    print(f"exact table: {kind} n={n} shots={nshots}", flush=True)
    for _ in range(2):  # the state is unchanged by a call
        idx, _, pr = st.sample([0], u)
        ref = np.searchsorted(orc.discrete_table(p), u, side="left")
        assert np.array_equal(idx, ref.astype(np.uint64))
        assert np.array_equal(pr, p[ref])


@pytest.mark.parametrize("n,nshots", [(2, 1025), (10, 1024), (10, 1025), (11, 1025), (13, 4096), (13, 4097),
                                      (17, 5000)])
def test_search_by_number_of_shots(qa, orc, n, nshots):
    """The error-bounded search's two ways through a chunk, at the shot
    counts where one takes over: indices equal the oracle's table."""
    rng = np.random.default_rng(n + nshots)
    psi = make_state("random", n, rng)
    p = orc.probs(psi)
    u = rng.random(nshots)
    print(f"search: n={n} shots={nshots}", flush=True)
    idx, _, pr = qa.State.from_array(psi, [2] * n).sample([0], u)
    ref = np.searchsorted(orc.discrete_table(p), u, side="left")
    assert np.array_equal(idx, ref.astype(np.uint64)) and np.array_equal(pr, p[ref])
