"""The pair-fused programs of the tile kernel hold select ops: a product that
joined an X under a lane or tile condition, kept in two versions (OP_U1S,
OP_U2S).  CPU: the circuits below give every kind the kernel has a case for,
and none that it has not (tests/cpp/tile_ops_check.cpp).  GPU: the same
circuits against the oracle, 1e-12 in complex128 and 5e-6 in complex64 (about
200 products of unit columns per amplitude, rounded to 2^-53 and 2^-24)."""
import os
import subprocess

import numpy as np
import pytest

from helpers import randket

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# qubits, depth, seed, low_bits, max_ops
CIRCUITS = [(14, 8, 1, 5, 64), (16, 10, 2, 3, 48), (17, 6, 3, 0, 200)]


def _layers(n, depth, seed):
    from qpp_amd import workloads
    return workloads.random_layers(n, depth, seed)


@pytest.fixture(scope="module")
def counter(tmp_path_factory):
    import qpp_amd
    qpp_amd.lib()
    exe = str(tmp_path_factory.mktemp("ops") / "tile_ops_check")
    lib = os.path.join(ROOT, "qpp_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                    os.path.join(HERE, "cpp", "tile_ops_check.cpp"), os.path.join(lib, "libqpp_amd.so"),
                    "-Wl,-rpath," + lib, "-Wl,-rpath,/opt/rocm/lib", "-Wl,--allow-shlib-undefined"], check=True)
    return exe


def test_every_select_op_occurs(counter):
    total = np.zeros(4, dtype=int)
    for n, depth, seed, low, max_ops in CIRCUITS:
        gates = _layers(n, depth, seed)
        text = [f"{n} {low} {max_ops} {len(gates)}"]
        for _, t, c, U in gates:
            mask = sum(1 << (n - 1 - q) for q in c)
            flat = np.asarray(U).reshape(-1, order="F")
            text.append(" ".join([str(len(t))] + [str(n - 1 - q) for q in t] + [str(mask), str(mask)] +
                                 [f"{v.real!r} {v.imag!r}" for v in flat.tolist()]))
        r = subprocess.run([counter], input="\n".join(text), capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        total += np.array([int(x) for x in r.stdout.split()])
    u1_lane, u1_tile, u2_tile, unknown = total
    assert u1_lane > 0 and u1_tile > 0 and u2_tile > 0 and unknown == 0, total


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n,depth,seed,low,max_ops", CIRCUITS)
def test_select_ops_vs_oracle(qa, orc, n, depth, seed, low, max_ops, dtype):
    dt, tol = (qa.C128, 1e-12) if dtype == "c128" else (qa.C64, 5e-6)
    gates = _layers(n, depth, seed)
    psi = randket(2 ** n, np.random.default_rng(seed))
    ref = psi
    for _, t, c, U in gates:
        ref = orc.applyCTRL(ref, U, c, t, 2) if c else orc.apply(ref, U, t, 2)
    st = qa.State.from_array(psi, [2] * n, dtype=dt)
    qa.Program(n, gates, dtype=dt, low_bits=low, max_ops=max_ops).run(st)
    assert np.max(np.abs(np.asarray(st.download()).astype(np.complex128) - ref)) <= tol
