"""Specialised pass kernels (qs_program_compile_native): every pass of a
tile program generated as its own kernel and compiled with hipRTC.  Checked
against the oracle applied gate by gate (complex128 <= 1e-12) on circuits
with every op kind the passes hold -- dense and diagonal 1-qubit gates,
dense 2-qubit gates, controls on register, thread and out-of-tile bits,
shifted controls, fans -- on kets and density matrices, with few
persistent workgroups walking many tiles, and at the benchmark's full size
(forward then inverse returns to |0...0>)."""
import numpy as np
import pytest

from helpers import haar, randket, randrho
from test_gpu_fused import maxabs, mixed_circuit, oracle_run

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("n", [12, 13, 16])
def test_native_mixed_gates_vs_oracle(qa, orc, n):
    qc = mixed_circuit(qa, n, 3, seed=300 + n)
    rng = np.random.default_rng(n + 5)
    psi = randket(2 ** n, rng)
    st = qa.State.from_array(psi, [2] * n)
    p = qa.Program(qc).compile_native()
    print(f"native n={n} {p.info()} kernel {p.kernel_name()}", flush=True)
    p.run(st)
    assert maxabs(st.download(), oracle_run(orc, psi, qc)) <= TOL


@pytest.mark.parametrize("n", [6, 7])
def test_native_rho_vs_oracle(qa, orc, n):
    qc = mixed_circuit(qa, n, 2, seed=400 + n)
    rng = np.random.default_rng(n + 6)
    rho = randrho(2 ** n, rng)
    st = qa.State.from_array(rho, [2] * n)
    qa.Program(qc, kind=qa.RHO).compile_native().run(st)
    assert maxabs(st.download(), oracle_run(orc, rho, qc)) <= TOL


def test_native_layouts_and_many_tiles(qa, orc):
    """Layout options that change which phases load, remap and store
    directly, with few persistent workgroups per pass (each walks many
    tiles, so prefetch, LDS layout changes and stores of consecutive tiles
    interleave)."""
    n = 17
    qc = mixed_circuit(qa, n, 3, seed=17)
    rng = np.random.default_rng(18)
    psi = randket(2 ** n, rng)
    ref = oracle_run(orc, psi, qc)
    for low, maxops, grid in ((0, 64, 5), (3, 8, 3), (6, 48, 64), (5, 200, 0)):
        print(f"native layout low={low} max_ops={maxops} grid={grid}", flush=True)
        st = qa.State.from_array(psi, [2] * n)
        qa.Program(qc, low_bits=low, max_ops=maxops, grid_cap=grid).compile_native().run(st)
        assert maxabs(st.download(), ref) <= TOL, (low, maxops, grid)


def test_native_c64_and_equal_to_tile_kernel(qa, orc):
    from qpp_amd import workloads
    n = 16
    gates = workloads.random_layers(n, 6, seed=9)
    qc = qa.QCircuit.from_gates(n, gates)
    psi = np.zeros(2 ** n, dtype=complex)
    psi[0] = 1
    ref = oracle_run(orc, psi, qc)
    a = qa.State.from_array(psi, [2] * n, dtype=qa.C64)
    qa.Program(qc, dtype=qa.C64).compile_native().run(a)
    out = a.download().astype(np.complex128)
    assert maxabs(out, ref) <= 5e-6 and 1 - abs(np.vdot(ref, out)) ** 2 <= 1e-6
    # the same complex products in the same order as the tile kernel
    b = qa.State.from_array(psi, [2] * n, dtype=qa.C64)
    qa.Program(qc, dtype=qa.C64).run(b)
    assert maxabs(out, b.download()) <= 1e-6


def test_native_rho_channels_bit_program(qa):
    """The density-matrix pipeline's gates and Kraus superoperators as one
    bit-level program: specialised kernels equal the tile kernel."""
    from qpp_amd import workloads
    n = 6
    rho, ops, _, _, _ = workloads.dm_pipeline(n, 3, seed=5)
    a = qa.State.from_array(rho, [2] * n)
    b = qa.State.from_array(rho, [2] * n)
    workloads.dm_program(qa, n, ops).compile().compile_native().run(a)
    workloads.dm_program(qa, n, ops).compile().run(b)
    assert maxabs(a.download(), b.download()) <= TOL


def test_native_needs_reg_bits_4(qa):
    from qpp_amd import workloads
    p = qa.Program(12, workloads.random_layers(12, 2, 1), reg_bits=3)
    with pytest.raises(qa.NotImplemented_):
        p.compile_native()


def test_native_full_size_circuit_and_inverse(qa):
    """The 30-qubit depth-40 benchmark circuit and its inverse through
    specialised kernels (complex128): back to |0...0> within 1e-12."""
    from qpp_amd import workloads
    n = 30
    gates = workloads.random_layers(n, 40, seed=30)
    inv = [(k, t, c, np.asarray(U).conj().T) for k, t, c, U in reversed(gates)]
    st = qa.State([2] * n)
    st.set_basis(0)
    qa.Program(n, gates, reg_bits=4, low_bits=3, max_ops=48).compile_native().run(st)
    assert abs(st.norm2() - 1) < 1e-12
    qa.Program(n, inv, reg_bits=4, low_bits=3, max_ops=48).compile_native().run(st)
    ref = qa.State([2] * n)
    ref.set_basis(0)
    r = st.compare(ref)
    assert r["infidelity"] < 1e-12 and r["max_abs"] < 1e-10, r


def test_native_split_layout_changes_vs_oracle(qa, orc):
    """Layout changes split in halves on a wave bit, a lane bit and a
    register bit (complex128; the passes whose changes all split run at half
    the LDS) and moved whole (complex64 keeps whole changes): circuits where
    every form occurs, against the oracle."""
    from qpp_amd import workloads
    seen = dict.fromkeys(("whole", "wave_split", "lane_split", "register_split", "half_lds_passes"), 0)
    for n, seed, low, maxops, dt in ((13, 1, 3, 16, qa.C128), (14, 2, 3, 48, qa.C128),
                                     (16, 1, 5, 48, qa.C128), (14, 3, 3, 48, qa.C64)):
        qc = qa.QCircuit.from_gates(n, workloads.random_layers(n, 12, seed))
        psi = randket(2 ** n, np.random.default_rng(seed + 50))
        st = qa.State.from_array(psi, [2] * n, dtype=dt)
        p = qa.Program(qc, dtype=dt, low_bits=low, max_ops=maxops).compile_native()
        stats = p.native_stats()
        print(f"native splits n={n} seed={seed} low={low} max_ops={maxops} dtype={dt}: {stats}", flush=True)
        p.run(st)
        tol = TOL if dt == qa.C128 else 5e-6
        assert maxabs(st.download().astype(np.complex128), oracle_run(orc, psi, qc)) <= tol, (n, seed, stats)
        for k in seen:
            seen[k] += stats[k]
    assert all(v > 0 for v in seen.values()), seen


def test_native_sign_diagonals_vs_oracle(qa, orc):
    """Diagonal entries of +-1 (Z, CZ, multi-controlled Z) become sign flips:
    on register bits, under lane and tile conditions, and as per-lane and
    per-tile factors (targets on thread bits and outside the tile), for
    complex128 and complex64, against the oracle."""
    from qpp_amd import workloads
    Z = np.diag([1, -1]).astype(complex)
    for n, seed, dt in ((14, 5, qa.C128), (16, 6, qa.C128), (15, 7, qa.C64)):
        rng = np.random.default_rng(seed)
        gates = []
        for kind, t, c, U in workloads.random_layers(n, 8, seed):
            if c:
                gates.append(("cz", t, c, Z))
            elif rng.random() < 0.3:
                gates.append(("z", t, [], Z))
            else:
                gates.append((kind, t, c, U))
        for _ in range(n):  # doubly controlled Z on random qubits
            q = [int(v) for v in rng.choice(n, 3, replace=False)]
            gates.append(("ccz", [q[0]], q[1:], Z))
        qc = qa.QCircuit.from_gates(n, gates)
        psi = randket(2 ** n, rng)
        st = qa.State.from_array(psi, [2] * n, dtype=dt)
        p = qa.Program(qc, dtype=dt).compile_native()
        print(f"native sign diagonals n={n} dtype={dt}: {p.info()}", flush=True)
        p.run(st)
        tol = TOL if dt == qa.C128 else 5e-6
        assert maxabs(st.download().astype(np.complex128), oracle_run(orc, psi, qc)) <= tol, (n, seed)


def _channels(kind, p):
    """(Kraus operators, the 2x2 map of the two populations) of a channel
    that keeps populations apart from coherences."""
    from qpp_amd import workloads
    if kind == "damping":
        return ([np.diag([1, np.sqrt(1 - p)]).astype(complex),
                 np.array([[0, np.sqrt(p)], [0, 0]], dtype=complex)], [[1, p], [0, 1 - p]])
    return workloads.depolarizing_kraus(p), [[1 - 2 * p / 3, 2 * p / 3], [2 * p / 3, 1 - 2 * p / 3]]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("channels", [[("damping", 0.01)], [("depolarizing", 1e-6)],
                                      [("damping", 0.3), ("depolarizing", 1e-6), ("damping", 1e-4)]])
def test_native_small_populations(qa, channels, dtype):
    """Channels on a diagonal density matrix whose populations span 21 orders
    of magnitude: every one is a sum of non-negative products, so it stays
    non-negative and keeps its relative accuracy however small it is beside
    the others.  The reference acts on the populations in extended precision;
    per channel a superoperator entry is within 8 roundings of it (the Kraus
    operators' roots, products and sum, in FP64, and its rounding to the
    state's type), the 4-term product within 4."""
    n = 6
    dt, eps, ctype = (qa.C128, 2.0 ** -53, np.complex128) if dtype == "c128" else (qa.C64, 2.0 ** -24, np.complex64)
    pops = np.ones(1, dtype=np.longdouble)
    for q in range(n):
        pops = np.kron(pops, np.array([1, 10.0 ** -(q + 1)], dtype=np.longdouble))
    pops = np.real(pops.astype(ctype)).astype(np.longdouble)
    bp = qa.BitProgram(2 * n)
    ref = pops.reshape([2] * n)
    for kind, p in channels:
        for q in range(n):
            Ks, M = _channels(kind, p)
            bp.rho_channel(Ks, q, n)
            ref = np.moveaxis(np.tensordot(np.array(M, dtype=np.longdouble), ref, axes=(1, q)), 0, q)
    ref = ref.reshape(-1)
    bp.compile(dtype=dt)
    tol = 12 * eps * n * len(channels)
    for native in (False, True):
        st = qa.State.from_array(np.diag(pops.astype(ctype)), [2] * n, dtype=dt)
        if native:
            bp.compile_native()
        bp.run(st)
        got = np.asarray(st.download())
        d = np.real(np.diag(got)).astype(np.longdouble)
        assert d.min() >= 0, (native, d.min())
        err = float(np.max(np.abs(d - ref) / ref))
        print(f"small populations {channels} {dtype} native={native}: relative error {err:.2e}", flush=True)
        assert err <= tol, (native, err, tol)
        assert not np.any(got - np.diag(np.diag(got)))


@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_bit_program_superoperators_vs_oracle(qa, orc, dtype):
    """Dense 4x4s of every kind a density-matrix program holds (depolarizing
    and amplitude damping superoperators, which mix populations one way, SWAP
    and Haar gates), some under controls that land on register, lane and
    out-of-tile bits, against the oracle applied op by op: specialised
    kernels, the tile kernel's fused program and its unfused one (reg_bits
    3).  The superoperators are within a factor 2 of norm 1, so the error is
    measured against the result's largest amplitude."""
    nb = 14
    rng = np.random.default_rng(77)
    swap = np.eye(4)[[0, 2, 1, 3]].astype(complex)
    bp, ops = qa.BitProgram(nb), []
    for i in range(60):
        bits = [int(b) for b in rng.permutation(nb)[:5]]
        kind = i % 5
        if kind < 2:
            Ks, _ = _channels("damping" if kind else "depolarizing", 0.05)
            M = sum(np.kron(K.conj(), K) for K in Ks)
        else:
            M = {2: swap, 3: haar(4, rng), 4: haar(2, rng)}[kind]
        nt = 1 if kind == 4 else 2
        ctrl = bits[2:2 + int(rng.integers(0, 4))]
        shift = [int(s) for s in rng.integers(0, 2, len(ctrl))]
        bp.gate(M, bits[:nt], sum(1 << c for c in ctrl), sum(1 << c for c, s in zip(ctrl, shift) if not s))
        ops.append((M, [nb - 1 - b for b in bits[:nt]], [nb - 1 - c for c in ctrl], shift))
    dt, tol = (qa.C128, 1e-12) if dtype == "c128" else (qa.C64, 1e-5)
    psi = randket(2 ** nb, rng)
    ref = psi
    for M, t, c, shift in ops:
        ref = orc.applyCTRL(ref, M, c, t, 2, shift) if c else orc.apply(ref, M, t, 2)
    for name in ("unfused", "fused", "specialised"):
        bp.compile(dtype=dt, reg_bits=3 if name == "unfused" else 4)
        if name == "specialised":
            bp.compile_native()
        st = qa.State.from_array(psi, [2] * nb, dtype=dt)
        bp.run(st)
        err = maxabs(np.asarray(st.download()).astype(np.complex128), ref) / np.max(np.abs(ref))
        print(f"superoperators {dtype} {name}: {err:.2e}", flush=True)
        assert err <= tol, (name, err)


@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_native_rho_pipeline_vs_oracle(qa, orc, dtype):
    """The density-matrix pipeline's circuit through the specialised and the
    tile kernel against the oracle, gate by gate and channel by channel."""
    from qpp_amd import workloads
    n = 6
    rho, ops, _, _, _ = workloads.dm_pipeline(n, 3, seed=5)
    ref = rho
    for kind, q, M in ops:
        if kind == "kraus":
            ref = orc.apply_kraus(ref, M, q, 2)
        elif kind == "cz":
            ref = orc.applyCTRL(ref, M, [q[0]], [q[1]], 2)
        else:
            ref = orc.apply(ref, M, q, 2)
    dt, tol = (qa.C128, TOL) if dtype == "c128" else (qa.C64, 5e-6)
    for native in (False, True):
        p = workloads.dm_program(qa, n, ops).compile(dtype=dt)
        if native:
            p.compile_native()
        st = qa.State.from_array(rho, [2] * n, dtype=dt)
        p.run(st)
        assert maxabs(np.asarray(st.download()).astype(np.complex128), ref) <= tol, native
