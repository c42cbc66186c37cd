"""The work a user of qpp_amd has it do, as cases that can be timed and checked.

Each case is one pass through the public Python entry points on device-resident
states: qpp's functions applied call by call (gates, controlled gates,
channels, maps, sampling and measurement), circuits compiled into fused passes,
the engine's execute loop and batches of noisy trajectories.  Sizes are those
of the repository's own benchmark and tests, and what lies between them.

`layout` seeds what a program fixes once (which gate acts on which subsystem,
the permutation, the targets); the seed given to `prepare` makes the data: the
state, the gate matrices, the uniforms and the engine seeds.
"""
import math
import random

import numpy as np
import torch

import qpp_amd as qa

DTYPES = {"c128": (qa.C128, 16, torch.complex128, "<c16"), "c64": (qa.C64, 8, torch.complex64, "<c8")}
X = np.array([[0, 1], [1, 0]], dtype=complex)
Z = np.diag([1.0, -1.0]).astype(complex)
NOISE = 1e-3  # depolarizing probability per qubit, the trajectory benchmark's


def listed():
    return [
        # interactive and test-sized use: a layer on a small register, call by
        # call, where each call's latency is what counts
        {"name": "gates small ket", "kind": "gates", "n": 10, "dtype": "c128", "count": 24, "kmax": 3, "layout": 1},
        # qpp::apply / applyCTRL on a large ket one call at a time, dense
        # gates of 1 to 3 qubits, in the reference's precision
        {"name": "gates large ket c128", "kind": "gates", "n": 25, "dtype": "c128", "count": 12, "kmax": 3, "layout": 2},
        # the same in complex64 up to 5-qubit dense gates (block gates)
        {"name": "gates large ket c64", "kind": "gates", "n": 28, "dtype": "c64", "count": 12, "kmax": 5, "layout": 3},
        # qpp::apply on a density matrix: gates and noise channels call by call
        {"name": "gates and channels rho", "kind": "rho", "n": 11, "dtype": "c128", "count": 12, "layout": 4},
        # a random circuit compiled once and run many times (variational
        # loops, the headline benchmark), passes specialised
        {"name": "circuit compiled", "kind": "circuit", "n": 28, "dtype": "c128", "depth": 12, "native": True, "layout": 5},
        # a noisy density-matrix circuit compiled into fused passes
        {"name": "rho circuit compiled", "kind": "rho_circuit", "n": 12, "dtype": "c128", "depth": 5, "layout": 6},
        # QEngine(qc, seed).execute(shots): a circuit met once, its gates, its
        # register measured and 1024 shots sampled
        {"name": "engine shots", "kind": "engine", "n": 22, "dtype": "c128", "depth": 20, "measured": 12, "shots": 1024, "layout": 7},
        # sampling and projective measurement of a large state
        {"name": "sample and measure", "kind": "measure", "n": 24, "dtype": "c128", "shots": 1024, "targets": 4, "destructive": False, "layout": 8},
        # partial trace, partial transpose and permutation of a density matrix
        {"name": "maps rho", "kind": "maps_rho", "n": 12, "dtype": "c128", "traced": 6, "layout": 9},
        # reduced states and permutations of a large ket
        {"name": "maps ket", "kind": "maps_ket", "n": 24, "dtype": "c128", "kept": 8, "layout": 10},
        # qutrits: gates, controlled gates, permutation and partial trace
        {"name": "qudits", "kind": "qudits", "n": 14, "d": 3, "dtype": "c128", "layout": 11},
        # noisy trajectories of the benchmark's sizes in one launch
        {"name": "trajectories", "kind": "trajectories", "n": 16, "wide": 20, "narrow_count": 192, "wide_count": 16,
         "dtype": "c128", "depth": 30, "layout": 12},
    ]


def draw(rng):
    layout = rng.randrange(1 << 30)
    kind = rng.choice(["gates", "gates", "gates", "rho", "circuit", "rho_circuit", "engine", "measure", "measure",
                       "maps_rho", "maps_ket", "qudits", "trajectories"])
    dtype = rng.choice(["c128", "c64"])
    c128 = dtype == "c128"
    if kind == "gates":
        n = rng.randint(6, 26 if c128 else 28)
        return {"kind": kind, "n": n, "dtype": dtype, "count": rng.randint(6, 24) if n < 22 else rng.randint(4, 12),
                "kmax": rng.randint(2, 4 if c128 else 5), "layout": layout}
    if kind == "rho":
        return {"kind": kind, "n": rng.randint(4, 12), "dtype": dtype, "count": rng.randint(4, 12), "layout": layout}
    if kind == "circuit":
        return {"kind": kind, "n": rng.randint(14, 27), "dtype": dtype, "depth": rng.randint(3, 12),
                "native": rng.random() < 0.5, "layout": layout}
    if kind == "rho_circuit":
        return {"kind": kind, "n": rng.randint(7, 12), "dtype": dtype, "depth": rng.randint(2, 5), "layout": layout}
    if kind == "engine":
        n = rng.randint(8, 24)
        return {"kind": kind, "n": n, "dtype": dtype, "depth": rng.randint(4, 20), "measured": rng.randint(2, min(n, 12)),
                "shots": rng.choice([1, 100, 1000, 1024, 4096]), "layout": layout}
    if kind == "measure":
        n = rng.randint(8, 26)
        return {"kind": kind, "n": n, "dtype": dtype, "shots": rng.choice([1, 7, 100, 1024, 5000]),
                "targets": rng.randint(1, 6), "destructive": rng.random() < 0.5, "layout": layout}
    if kind == "maps_rho":
        n = rng.randint(4, 12)
        return {"kind": kind, "n": n, "dtype": dtype, "traced": rng.randint(1, n - 1), "layout": layout}
    if kind == "maps_ket":
        n = rng.randint(12, 26)
        return {"kind": kind, "n": n, "dtype": dtype, "kept": rng.randint(1, 9), "layout": layout}
    if kind == "qudits":
        d = rng.choice([3, 3, 4, 5])
        top = {3: 14, 4: 11, 5: 9}[d]
        return {"kind": kind, "n": rng.randint(4, top), "d": d, "dtype": dtype, "layout": layout}
    # final outcomes are compared one by one: complex128, where no shot sits
    # within rounding of a cumulative edge
    return {"kind": kind, "n": rng.randint(10, 16), "wide": rng.randint(18, 20), "narrow_count": rng.randint(16, 192),
            "wide_count": rng.randint(1, 16), "dtype": "c128", "depth": rng.randint(8, 30), "layout": layout}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Buffer:
    """A state's device memory for torch; the state lives as long as this."""

    def __init__(self, st):
        dt, _, _, ne = st.info()
        ptr = qa.c_void_p()
        qa._check(qa.lib().qs_state_device_ptr(st.handle, qa.byref(ptr)))
        self.state = st
        self.__cuda_array_interface__ = {"shape": (ne,), "typestr": "<c16" if dt == qa.C128 else "<c8",
                                         "data": (ptr.value, False), "strides": None, "version": 2}


def _tensor(st):
    """The state's amplitudes (density matrices column by column), no copy."""
    return torch.as_tensor(_Buffer(st), device="cuda")


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _ket(size, seed):
    v = torch.randn(size, dtype=torch.complex128, device="cuda", generator=_generator(seed))
    return v.div_(torch.linalg.vector_norm(v))


def _rho(D, seed):
    """0.9 |psi><psi| + 0.1 I / D, column-major, flat."""
    v = _ket(D, seed)
    r = torch.outer(v.conj(), v).mul_(0.9).reshape(-1)
    r[:: D + 1] += 0.1 / D
    return r


def _state(dims, kind, dtype, data):
    st = qa.State(dims, kind, DTYPES[dtype][0])
    qa.synchronize()
    _tensor(st).copy_(data)
    torch.cuda.synchronize()
    return st


def _haar(d, rng):
    z = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    q, r = np.linalg.qr(z)
    return q * (np.diag(r) / np.abs(np.diag(r)))


def _depolarizing(p):
    Y = np.array([[0, -1j], [1j, 0]])
    return [math.sqrt(1 - p) * np.eye(2, dtype=complex), math.sqrt(p / 3) * X, math.sqrt(p / 3) * Y, math.sqrt(p / 3) * Z]


def _damping(g):
    return [np.diag([1, math.sqrt(1 - g)]).astype(complex), np.array([[0, math.sqrt(g)], [0, 0]], dtype=complex)]


def _ket_ops(case):
    """(name, controls, targets, shift) of each call: mostly 1-qubit gates
    and CNOTs, some wider and multi-controlled ones."""
    rng, n = random.Random(case["layout"]), case["n"]
    names = ["u1", "cx", "u2", "u1", "ccu", "u3", "cx", "u1", "fan", "cu2", "u4", "u5"]
    names = [m for m in names if not (m[0] == "u" and int(m[1]) > case["kmax"])]
    ops = []
    for i in range(case["count"]):
        name = names[i % len(names)]
        nc = {"cx": 1, "ccu": 2, "cu2": 1, "fan": 1}.get(name, 0)
        nt = {"u1": 1, "u2": 2, "u3": 3, "u4": 4, "u5": 5, "cx": 1, "ccu": 1, "cu2": 2, "fan": 3}[name]
        q = rng.sample(range(n), nc + nt)
        ops.append((name, q[:nc], q[nc:], [rng.randrange(2) for _ in range(nc)] if name == "ccu" else None))
    return ops


def _matrices(case, seed):
    rng = np.random.default_rng(seed)
    return [X if name == "cx" else _haar(2 if name == "fan" else 2 ** len(t), rng) for name, _, t, _ in _ket_ops(case)]


def _rho_ops(case):
    rng, n = random.Random(case["layout"]), case["n"]
    names = ["u1", "dep", "cx", "damp", "u2", "dep", "u1", "dep2"]
    return [(names[i % len(names)], rng.sample(range(n), 2)) for i in range(case["count"])]


def _rho_matrices(case, seed):
    rng, out = np.random.default_rng(seed), []
    for name, _ in _rho_ops(case):
        if name == "dep":
            out.append(_depolarizing(float(rng.uniform(0.0005, 0.002))))
        elif name == "damp":
            out.append(_damping(float(rng.uniform(0.0005, 0.002))))
        elif name == "dep2":
            a, b = _depolarizing(float(rng.uniform(0.0005, 0.002))), _depolarizing(float(rng.uniform(0.0005, 0.002)))
            out.append([np.kron(x, y) for x in a for y in b])
        else:
            out.append(X if name == "cx" else _haar(4 if name == "u2" else 2, rng))
    return out


def _layers(n, depth, layout, seed, noisy=False):
    """Layers of a Haar gate on every qubit and CNOTs (noisy: CZ) on a random
    pairing: (targets, controls, matrix)."""
    where, rng, gates = random.Random(layout), np.random.default_rng(seed), []
    for _ in range(depth):
        gates += [([q], [], _haar(2, rng)) for q in range(n)]
        p = where.sample(range(n), n)
        gates += [([p[i + 1]], [p[i]], Z if noisy else X) for i in range(0, n - 1, 2)]
    return gates


def _circuit(n, gates, nc=0):
    qc = qa.QCircuit(n, nc)
    for t, c, U in gates:
        qc.CTRL(U, c, t) if c else qc.gate(U, t)
    return qc


def _ladder(n, depth, rng):
    gates = []
    for _ in range(depth):
        gates += [([q], [], _haar(2, rng)) for q in range(n)]
        gates += [([q + 1], [q], X) for q in range(n - 1)]
    return _circuit(n, gates, n).measure(list(range(n)), 0)


def _qudit_plan(case):
    rng, n = random.Random(case["layout"]), case["n"]
    return {"one": rng.sample(range(n), 2), "two": rng.sample(range(n), 2), "ctrl": rng.sample(range(n), 2),
            "perm": rng.sample(range(n), n), "trace": sorted(rng.sample(range(n), max(1, n - min(4, n // 2))))}


def _some(case, count, among=None):
    return random.Random(case["layout"]).sample(range(among or case["n"]), count)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, n, dtype = case["kind"], case["n"], case["dtype"]
    s = {"case": case, "kind": kind, "n": n}
    if kind == "gates":
        s["state"] = _state([2] * n, qa.KET, dtype, _ket(2 ** n, seed))
        s["calls"] = [(op, M) for op, M in zip(_ket_ops(case), _matrices(case, seed))]
    elif kind == "rho":
        s["state"] = _state([2] * n, qa.RHO, dtype, _rho(2 ** n, seed))
        s["calls"] = [(op, M) for op, M in zip(_rho_ops(case), _rho_matrices(case, seed))]
    elif kind == "circuit":
        s["state"] = _state([2] * n, qa.KET, dtype, _ket(2 ** n, seed))
        qc = _circuit(n, _layers(n, case["depth"], case["layout"], seed))
        s["program"] = qa.Program(qc, dtype=DTYPES[dtype][0], low_bits=3, max_ops=48, grid_cap=65536)
        if case["native"]:
            s["program"].compile_native()
    elif kind == "rho_circuit":
        s["state"] = _state([2] * n, qa.RHO, dtype, _rho(2 ** n, seed))
        bp, Ks = qa.BitProgram(2 * n), _depolarizing(NOISE)
        for t, c, U in _layers(n, case["depth"], case["layout"], seed, noisy=True):
            bp.rho_ctrl(U, c, t, n) if c else bp.rho_apply(U, t, n)
            for q in c + t:
                bp.rho_channel(Ks, q, n)
        s["program"] = bp.compile(dtype=DTYPES[dtype][0])
        bp.compile_native()
    elif kind == "engine":
        qc = _circuit(n, _layers(n, case["depth"], case["layout"], seed), case["measured"])
        s["circuit"] = qc.measure(list(range(case["measured"])), 0, destructive=False)
        s["seed"] = int(seed)
    elif kind == "measure":
        s["state"] = _state([2] * n, qa.KET, dtype, _ket(2 ** n, seed))
        rng = np.random.default_rng(seed)
        s["u"], s["v"] = rng.random(case["shots"]), float(rng.random())
    elif kind == "maps_rho":
        s["state"] = _state([2] * n, qa.RHO, dtype, _rho(2 ** n, seed))
    elif kind == "maps_ket":
        s["state"] = _state([2] * n, qa.KET, dtype, _ket(2 ** n, seed))
        s["half"] = _state([2] * (n // 2), qa.KET, dtype, _ket(2 ** (n // 2), seed + 1))
    elif kind == "qudits":
        d, rng = case["d"], np.random.default_rng(seed)
        s["state"] = _state([d] * n, qa.KET, dtype, _ket(d ** n, seed))
        s["U"], s["V"], s["W"] = _haar(d, rng), _haar(d * d, rng), _haar(d, rng)
    elif kind == "trajectories":
        rng = np.random.default_rng(case["layout"])
        s["batch"] = qa.Batch([_ladder(case["n"], case["depth"], rng), _ladder(case["wide"], case["depth"], rng)],
                              dtype=DTYPES[dtype][0])
        s["which"] = [0] * case["narrow_count"] + [1] * case["wide_count"]
        s["seeds"] = np.random.default_rng(seed).integers(1, 2 ** 31, len(s["which"]))
    return s


def run(s):
    case, kind, n = s["case"], s["kind"], s["n"]
    if kind == "gates":
        st = s["state"]
        for (name, c, t, shift), M in s["calls"]:
            if name == "fan":
                st.apply_ctrl_fan(M, c, t)
            elif c:
                st.apply_ctrl(M, c, t, shift)
            else:
                st.apply(M, t)
        return _tensor(st)
    if kind == "rho":
        st = s["state"]
        for (name, q), M in s["calls"]:
            if name == "cx":
                st.apply_ctrl(M, q[:1], q[1:])
            elif name in ("dep", "damp"):
                st.apply_kraus(M, q[:1])
            elif name == "dep2":
                st.apply_kraus(M, q)
            else:
                st.apply(M, q if name == "u2" else q[:1])
        return _tensor(st)
    if kind in ("circuit", "rho_circuit"):
        s["program"].run(s["state"])
        return _tensor(s["state"])
    if kind == "engine":
        e = qa.QEngine(s["circuit"], dtype=DTYPES[case["dtype"]][0], seed=s["seed"]).execute(case["shots"])
        hist = np.zeros(2 ** case["measured"], dtype=np.int64)
        for dits, count in e.get_stats().items():
            hist[int("".join(map(str, dits)), 2)] = count
        return {"hist": hist, "state": _tensor(e.get_state())}
    if kind == "measure":
        idx, _, pr = s["state"].sample(list(range(n)), s["u"])
        st = s["state"].clone()
        res, ps = st.measure_seq(_some(case, case["targets"]), s["v"], case["destructive"])
        return {"idx": idx.astype(np.int64), "probs": pr, "result": np.array(res), "result_probs": np.array(ps),
                "state": _tensor(st)}
    if kind == "maps_rho":
        st = s["state"]
        out = [st.ptrace(sorted(_some(case, case["traced"]))), st.ptranspose(_some(case, n // 3 + 1)),
               st.syspermute(_some(case, n))]
        return [_tensor(o) for o in out]
    if kind == "maps_ket":
        kept = _some(case, case["kept"])
        out = [s["state"].ptrace([q for q in range(n) if q not in kept]), s["state"].syspermute(_some(case, n)),
               s["half"].ptranspose(_some(case, n // 6 + 1, n // 2))]
        return [_tensor(o) for o in out]
    if kind == "qudits":
        st, p = s["state"], _qudit_plan(case)
        for q in p["one"]:
            st.apply(s["U"], [q])
        st.apply(s["V"], p["two"])
        st.apply_ctrl(s["W"], p["ctrl"][:1], p["ctrl"][1:])
        return [_tensor(st), _tensor(st.syspermute(p["perm"])), _tensor(st.ptrace(p["trace"]))]
    idx, pr = s["batch"].run(s["which"], s["seeds"], NOISE)
    return {"idx": idx.astype(np.int64), "probs": pr}


def work(case):
    """Bytes: a call on its own reads each amplitude it acts on once and
    writes it once; a compiled circuit reads and writes its state once.
    Operations: dense products (8 real ones per complex multiply-add)."""
    kind, n, z = case["kind"], case["n"], DTYPES[case["dtype"]][1]
    if kind == "gates":
        touched = [((3 if name == "fan" else 1) * 2.0 ** (n - len(c)), 2 if name == "fan" else 2 ** len(t))
                   for name, c, t, _ in _ket_ops(case)]
        return {"bytes": sum(2 * z * a for a, _ in touched), "flops": sum(8 * a * k for a, k in touched)}
    if kind == "rho":
        b = f = 0.0
        for name, _ in _rho_ops(case):
            a = 4.0 ** n * (0.75 if name == "cx" else 1)
            b += 2 * z * a
            f += 8 * a * {"cx": 1, "u2": 8, "dep2": 16}.get(name, 4)
        return {"bytes": b, "flops": f}
    if kind == "circuit":
        return {"bytes": 2 * z * 2.0 ** n, "flops": case["depth"] * n * 14 * 2.0 ** n}
    if kind == "rho_circuit":
        return {"bytes": 2 * z * 4.0 ** n, "flops": case["depth"] * n * 28 * 4.0 ** n}
    if kind == "engine":
        return {"bytes": 2 * z * 2.0 ** n, "flops": case["depth"] * n * 14 * 2.0 ** n}
    if kind == "measure":  # sampling reads the state, measuring reads it and writes the new one
        kept = 2.0 ** (n - case["targets"]) if case["destructive"] else 2.0 ** n
        return {"bytes": z * (2 * 2.0 ** n + kept), "flops": 3 * 2.0 ** n}
    if kind == "maps_rho":
        t = case["traced"]
        return {"bytes": z * (4.0 ** n / 2 ** t + 4.0 ** (n - t) + 4 * 4.0 ** n), "flops": 2 * 4.0 ** n / 2 ** t}
    if kind == "maps_ket":
        k, h = case["kept"], n // 2
        return {"bytes": z * (3 * 2.0 ** n + 4.0 ** k + 2.0 ** h + 4.0 ** h), "flops": 8 * 2.0 ** (n + k) + 6 * 4.0 ** h}
    if kind == "qudits":
        d, k = case["d"], n - len(_qudit_plan(case)["trace"])
        D = float(d) ** n
        return {"bytes": z * (2 * D * (3 + (d - 1) / d) + 2 * D + D + d ** (2 * k)),
                "flops": 8 * D * (2 * d + d * d + (d - 1)) + 8 * D * d ** k}
    a = case["narrow_count"] * 2.0 ** n, case["wide_count"] * 2.0 ** case["wide"]
    return {"bytes": z * sum(a), "flops": case["depth"] * 14 * (a[0] * n + a[1] * case["wide"])}


def tolerance(case):
    """What rounding in the case's own precision allows; whole results may
    differ where a uniform lies within rounding of a cumulative edge."""
    # measured against exact(): 2e-16 to 9e-15 in complex128 (the longest sums
    # are partial traces), 2e-7 in complex64 for a dozen gates
    rel = 2e-6 if case["dtype"] == "c64" else 5e-14
    if case["kind"] == "trajectories":
        return {"rel": 1e-10, "differ": 0.0}
    if case["kind"] == "engine":  # renormalised after each measured qubit
        return {"rel": 2 * rel, "differ": 0.01 if case["dtype"] == "c64" else 0.0}
    return {"rel": rel}


# ---------------------------------------------------------------------------
# the same results in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _apply(v, dims, U, axes, fixed=()):
    """U on the digits `axes` of the flat array v (in place), where the
    digits fixed = [(axis, value), ...] hold."""
    U = np.asarray(U)
    pinned = dict(fixed)
    shape, picks, run_ = [], [], 1
    for a, d in enumerate(dims):
        if a in pinned or a in axes:
            shape += [run_, d]
            picks.append(a)
            run_ = 1
        else:
            run_ *= d
    shape.append(run_)
    w = v.view(shape)

    def part(digits):
        x = w
        for j in range(len(picks) - 1, -1, -1):
            x = x.select(2 * j + 1, {**pinned, **digits}[picks[j]])
        return x

    combos = list(np.ndindex(*[dims[a] for a in axes]))
    ins = [part(dict(zip(axes, c))).clone() for c in combos]
    for r, c in enumerate(combos):
        o = torch.zeros_like(ins[r])
        for k, x in enumerate(ins):
            if U[r, k] != 0:
                o.add_(x, alpha=complex(U[r, k]))
        part(dict(zip(axes, c))).copy_(o)
        del o
    return v


def _permuted(v, dims, perm):
    """Output digit k is input digit perm[k]."""
    out = [dims[p] for p in perm]
    y = torch.arange(v.numel(), device=v.device)
    x = torch.zeros_like(y)
    for k, p in enumerate(perm):
        stride = math.prod(out[k + 1:])
        x += y // stride % out[k] * math.prod(dims[p + 1:])
    return v[x]


def _reduced(v, dims, trace):
    """tr_trace |v><v|, column-major, flat."""
    keep = [q for q in range(len(dims)) if q not in trace]
    M = _permuted(v, dims, keep + list(trace)).view(math.prod(dims[q] for q in keep), -1)
    return (M @ M.conj().T).T.reshape(-1).contiguous()


def _draws(p, u):
    c = torch.cumsum(p, 0)
    c = c / c[-1]
    c[-1] = 1
    return torch.searchsorted(c, torch.as_tensor(u, device=p.device))


def _exact_measure(case, seed):
    n, rng = case["n"], np.random.default_rng(seed)
    v = _rounded(case, _ket(2 ** n, seed))
    p = v.real.square() + v.imag.square()
    u, w = rng.random(case["shots"]), float(rng.random())
    idx, one = _draws(p, u), int(_draws(p, [w])[0])
    targets = _some(case, case["targets"])
    res = [one >> (n - 1 - t) & 1 for t in targets]
    # the order the results are projected in: as given, or when destructive
    # from the last subsystem down
    order = sorted(range(len(targets)), key=lambda k: -targets[k]) if case["destructive"] else range(len(targets))
    at, ps, keep = torch.arange(2 ** n, device=v.device), [0.0] * len(targets), None
    before = torch.ones((), dtype=p.dtype, device=p.device)
    for k in order:
        hit = (at >> (n - 1 - targets[k]) & 1) == res[k]
        keep = hit if keep is None else keep & hit
        now = p[keep].sum()
        ps[k], before = float(now / before), now
    out = v[keep] if case["destructive"] else torch.where(keep, v, 0)
    return {"idx": idx.cpu().numpy(), "probs": p[idx].cpu().numpy(), "result": np.array(res), "result_probs": np.array(ps),
            "state": out / before.sqrt()}


def _rounded(case, data):
    """The inputs as the state holds them, in 64 bits."""
    return data if case["dtype"] == "c128" else data.to(torch.complex64).to(torch.complex128)


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "gates":
        v = _rounded(case, _ket(2 ** n, seed))
        for (name, c, t, shift), U in zip(_ket_ops(case), _matrices(case, seed)):
            fixed = [(a, 1 - b) for a, b in zip(c, shift or [0] * len(c))]
            for axes in ([[q] for q in t] if name == "fan" else [t]):
                _apply(v, [2] * n, U, axes, fixed)
        return v
    if kind in ("rho", "rho_circuit"):
        v, dims = _rounded(case, _rho(2 ** n, seed)), [2] * (2 * n)  # digits: columns, then rows

        def both(U, t, c=()):
            _apply(v, dims, np.conj(U), list(t), [(a, 1) for a in c])
            _apply(v, dims, U, [n + q for q in t], [(n + a, 1) for a in c])

        def channel(Ks, t):
            _apply(v, dims, sum(np.kron(K.conj(), K) for K in Ks), list(t) + [n + q for q in t])

        if kind == "rho":
            for (name, q), M in zip(_rho_ops(case), _rho_matrices(case, seed)):
                if name in ("dep", "damp"):
                    channel(M, q[:1])
                elif name == "dep2":
                    channel(M, q)
                else:
                    both(M, q[1:] if name == "cx" else q if name == "u2" else q[:1], q[:1] if name == "cx" else ())
            return v
        for t, c, U in _layers(n, case["depth"], case["layout"], seed, noisy=True):
            both(U, t, c)
            for q in c + t:
                channel(_depolarizing(NOISE), [q])
        return v
    if kind == "circuit":
        v = _rounded(case, _ket(2 ** n, seed))
        for t, c, U in _layers(n, case["depth"], case["layout"], seed):
            _apply(v, [2] * n, U, t, [(a, 1) for a in c])
        return v
    if kind == "measure":
        return _exact_measure(case, seed)
    if kind == "maps_rho":
        v = _rounded(case, _rho(2 ** n, seed))
        trace, swap, perm = sorted(_some(case, case["traced"])), _some(case, n // 3 + 1), _some(case, n)
        keep = [q for q in range(n) if q not in trace]
        w = _permuted(v, [2] * (2 * n), keep + [n + q for q in keep] + trace + [n + q for q in trace])
        traced = w.view(4 ** len(keep), 2 ** len(trace), 2 ** len(trace)).diagonal(dim1=1, dim2=2).sum(-1)
        rows = [q if q in swap else n + q for q in range(n)]
        cols = [n + q if q in swap else q for q in range(n)]
        return [traced, _permuted(v, [2] * (2 * n), cols + rows), _permuted(v, [2] * (2 * n), perm + [n + q for q in perm])]
    if kind == "maps_ket":
        v, h = _rounded(case, _ket(2 ** n, seed)), n // 2
        w = _rounded(case, _ket(2 ** h, seed + 1))
        kept, swap = _some(case, case["kept"]), _some(case, n // 6 + 1, h)
        r = torch.outer(w.conj(), w).reshape(-1)
        cols = [h + q if q in swap else q for q in range(h)]
        rows = [q if q in swap else h + q for q in range(h)]
        return [_reduced(v, [2] * n, [q for q in range(n) if q not in kept]), _permuted(v, [2] * n, _some(case, n)),
                _permuted(r, [2] * (2 * h), cols + rows)]
    if kind == "qudits":
        d, rng, p = case["d"], np.random.default_rng(seed), _qudit_plan(case)
        dims, v = [d] * n, _rounded(case, _ket(d ** n, seed))
        U, V, W = _haar(d, rng), _haar(d * d, rng), _haar(d, rng)
        for q in p["one"]:
            _apply(v, dims, U, [q])
        _apply(v, dims, V, p["two"])
        for r in range(1, d):  # control digit r: the r-th power
            _apply(v, dims, np.linalg.matrix_power(W, r), p["ctrl"][1:], [(p["ctrl"][0], r)])
        return [v, _permuted(v, dims, p["perm"]), _reduced(v, dims, p["trace"])]
    return None
