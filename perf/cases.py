"""Workloads of the state-vector engine, from the smallest calls to the largest.

Each case is the work a user's program does through the public entry points
once its circuit, parameters and device buffers exist:

* ``gates``    -- rotations and a CX chain (GHZ-like) applied gate by gate with
                  ``functionals.apply`` (the reference's per-gate loop);
* ``program``  -- a whole circuit through ``functionals.Program``: random
                  layered circuits fused into blocks of at most 5 qubits, and
                  lists of all gate classes run unfused;
* ``adjoint``  -- energy and gradient of a hardware-efficient ansatz by
                  ``Program.adjoint`` (training of variational circuits);
* ``params``   -- energies of many parameter sets of one ansatz
                  (``batch.ParameterBatch``);
* ``circuits`` -- different circuits of uneven qubit counts as one batch
                  (``cbatch.circuit_batch``);
* ``qaoa``     -- energies and gradients of a batch of MaxCut instances
                  (``qaoa.qaoa_batch``);
* ``sample``   -- shots from a prepared state with numpy's choice semantics
                  (``functionals.sample``);
* ``simulate`` -- an OpenQASM 3 program through ``StateVectorSimulator.run``.

Circuits are drawn here as plain (name, targets, angles, matrix) tuples; the
64-bit values are computed from the same tuples with torch alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from snuqs_amd import _C
from snuqs_amd.batch import ParameterBatch
from snuqs_amd.cbatch import circuit_batch
from snuqs_amd.qaoa import qaoa_batch
from snuqs_amd.simulator import StateVectorSimulator
from snuqs_amd.transpile import fuse_operations

G = _C.operation.gate_operations
F = _C.functionals


def listed():
    return [
        # a 20-qubit entangled state in complex128, one apply call per gate: the
        # reference's own way of running a circuit, at its test size
        {"name": "chain_20q_c128", "kind": "gates", "n": 20, "dtype": "complex128"},
        # a small circuit replayed from a captured graph: latency of launches
        {"name": "layered_14q_c64_graph", "kind": "program", "style": "layered", "n": 14, "depth": 10,
         "dtype": "complex64", "fuse": 5, "graph": True},
        # an ordinary circuit, odd qubit count (a state that fits the caches)
        {"name": "layered_23q_c64", "kind": "program", "style": "layered", "n": 23, "depth": 12,
         "dtype": "complex64", "fuse": 5, "graph": False},
        # the benchmark circuit family at its 30 qubits (8 GiB of state)
        {"name": "layered_30q_c64", "kind": "program", "style": "layered", "n": 30, "depth": 10,
         "dtype": "complex64", "fuse": 5, "graph": False},
        # a large complex128 state, odd qubit count (2 GiB)
        {"name": "layered_27q_c128", "kind": "program", "style": "layered", "n": 27, "depth": 8,
         "dtype": "complex128", "fuse": 5, "graph": False},
        # every gate class, unfused: phases, diagonals, permutations, dense
        # gates on low and high bits, controls (the random-circuit test)
        {"name": "mixed_25q_c64_unfused", "kind": "program", "style": "mixed", "n": 25, "depth": 6,
         "dtype": "complex64", "fuse": 0, "graph": False},
        # 24-qubit ansatz, 384 parameters, 64 Pauli strings: one training step
        {"name": "adjoint_24q_c64", "kind": "adjoint", "n": 24, "layers": 8, "terms": 64,
         "dtype": "complex64", "checkpoints": 4},
        # 64 parameter sets of a 20-qubit ansatz: one generation of a
        # gradient-free optimiser or a parameter-shift batch
        {"name": "params_64x20q_c64", "kind": "params", "n": 20, "layers": 8, "sets": 64,
         "terms": 64, "dtype": "complex64"},
        # an ensemble of different circuits, 12-22 qubits
        {"name": "circuits_48_c64", "kind": "circuits", "lo": 12, "hi": 22, "count": 48,
         "depth": 10, "dtype": "complex64"},
        # MaxCut instances of 12-24 qubits, p = 4: energies and gradients
        {"name": "qaoa_64_c64", "kind": "qaoa", "lo": 12, "hi": 24, "count": 64, "p": 4,
         "dtype": "complex64"},
        # 100,000 shots from a 26-qubit complex64 state
        {"name": "sample_26q_c64", "kind": "sample", "n": 26, "shots": 100000, "dtype": "complex64"},
        # the Braket entry point end to end: source text in, results out
        {"name": "simulate_16q_c128", "kind": "simulate", "n": 16, "depth": 6, "dtype": "complex128"},
    ]


def draw(rng):
    kind = rng.choice(["gates", "program", "program", "program", "program", "program", "adjoint",
                       "params", "circuits", "qaoa", "sample", "simulate"])
    dt = rng.choice(["complex64", "complex64", "complex128"])
    if kind == "gates":
        return {"kind": kind, "n": rng.randint(10, 26), "dtype": dt}
    if kind == "program":
        style = rng.choice(["layered", "layered", "mixed", "u_cx"])
        fuse = rng.choice([5, 5, 4, 0])
        top = (28 if fuse else 26) - (dt == "complex128")
        n = rng.randint(12, top)
        depth = rng.randint(3, 12)
        return {"kind": kind, "style": style, "n": n, "depth": depth, "dtype": dt, "fuse": fuse,
                "graph": rng.random() < 0.4}
    if kind == "adjoint":
        return {"kind": kind, "n": rng.randint(12, 24), "layers": rng.randint(2, 8),
                "terms": rng.randint(8, 64), "dtype": dt, "checkpoints": rng.choice([0, 2, 4])}
    if kind == "params":
        return {"kind": kind, "n": rng.randint(10, 19), "layers": rng.randint(2, 8),
                "sets": rng.randint(5, 64), "terms": rng.randint(8, 64), "dtype": dt}
    if kind == "circuits":
        lo = rng.randint(6, 14)
        return {"kind": kind, "lo": lo, "hi": lo + rng.randint(4, 8), "count": rng.randint(8, 60),
                "depth": rng.randint(4, 10), "dtype": dt}
    if kind == "qaoa":
        lo = 2 * rng.randint(4, 8)
        return {"kind": kind, "lo": lo, "hi": lo + 2 * rng.randint(1, 4),
                "count": rng.randint(8, 64), "p": rng.randint(1, 5), "dtype": dt}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(12, 26), "shots": int(10 ** rng.uniform(2, 6)),
                "dtype": dt}
    return {"kind": kind, "n": rng.randint(6, 20), "depth": rng.randint(2, 6), "dtype": dt}


# --------------------------------------------------------------------------
# circuits as plain tuples
# --------------------------------------------------------------------------
_R2 = math.sqrt(0.5)
_FIXED = {
    "h": np.array([[_R2, _R2], [_R2, -_R2]]),
    "x": np.array([[0, 1], [1, 0]]),
    "y": np.array([[0, -1j], [1j, 0]]),
    "z": np.diag([1, -1]),
    "s": np.diag([1, 1j]),
    "t": np.diag([1, np.exp(0.25j * math.pi)]),
    "cx": np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]]),
    "cz": np.diag([1, 1, 1, -1]),
    "swap": np.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]]),
    "iswap": np.array([[1, 0, 0, 0], [0, 0, 1j, 0], [0, 1j, 0, 0], [0, 0, 0, 1]]),
    "ccx": np.eye(8)[[0, 1, 2, 3, 4, 5, 7, 6]],
}
_TARGETS = {"h": 1, "x": 1, "y": 1, "z": 1, "s": 1, "t": 1, "cx": 2, "cz": 2, "swap": 2,
            "iswap": 2, "ccx": 3, "rx": 1, "ry": 1, "rz": 1, "phase": 1, "cphase": 2, "xx": 2,
            "zz": 2}
_CTOR = {"h": G.Hadamard, "x": G.PauliX, "y": G.PauliY, "z": G.PauliZ, "s": G.S, "t": G.T,
         "cx": G.CX, "cz": G.CZ, "swap": G.Swap, "iswap": G.ISwap, "ccx": G.CCNot, "rx": G.RotX,
         "ry": G.RotY, "rz": G.RotZ, "phase": G.PhaseShift, "cphase": G.CPhaseShift, "xx": G.XX,
         "zz": G.ZZ}


def _matrix(name, a):
    if name in _FIXED:
        return _FIXED[name].astype(np.complex128)
    c, s = math.cos(a / 2), math.sin(a / 2)
    if name == "rx":
        return np.array([[c, -1j * s], [-1j * s, c]])
    if name == "ry":
        return np.array([[c, -s], [s, c]], dtype=np.complex128)
    if name == "rz":
        return np.diag(np.exp([-0.5j * a, 0.5j * a]))
    if name == "phase":
        return np.diag([1, np.exp(1j * a)])
    if name == "cphase":
        return np.diag([1, 1, 1, np.exp(1j * a)])
    if name == "zz":
        return np.diag(np.exp(np.array([-0.5j, 0.5j, 0.5j, -0.5j]) * a))
    return c * np.eye(4) - 1j * s * np.eye(4)[::-1]  # xx


def _gate(name, targets, angle=None):
    return name, [int(t) for t in targets], angle, _matrix(name, angle)


def _haar(d, rng):
    z = (rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))) * _R2
    q, r = np.linalg.qr(z)
    return q * (np.diagonal(r) / np.abs(np.diagonal(r)))


def _circuit(style, n, depth, rng):
    """Layered: Haar 2-qubit gates on a random pairing, then RotZ on every
    qubit.  u_cx: Haar 1-qubit gates, then CX on a random pairing.  mixed: H
    on every qubit, then depth * n gates of random kinds and targets."""
    out = []
    if style == "mixed":
        out = [_gate("h", [q]) for q in range(n)]
        kinds = sorted(_TARGETS)
        for _ in range(depth * n):
            k = kinds[int(rng.integers(len(kinds)))]
            out.append(_gate(k, rng.permutation(n)[:_TARGETS[k]], float(rng.uniform(0, 2 * math.pi))))
        return out
    for _ in range(depth):
        if style == "u_cx":
            out += [("unitary", [q], None, _haar(2, rng)) for q in range(n)]
        p = rng.permutation(n)
        for w in range(n // 2):
            t = [int(p[2 * w]), int(p[2 * w + 1])]
            out.append(_gate("cx", t) if style == "u_cx" else ("unitary", t, None, _haar(4, rng)))
        if style == "layered":
            out += [_gate("rz", [q], float(rng.uniform(0, 2 * math.pi))) for q in range(n)]
    return out


def _ansatz(n, layers, thetas):
    """Layers of RotY and RotZ on every qubit and a ring of CZ; the parameter
    of each gate (or None)."""
    gates, params, p = [], [], 0
    for _ in range(layers):
        for name in ("ry", "rz"):
            for q in range(n):
                gates.append(_gate(name, [q], float(thetas[p])))
                params.append(p)
                p += 1
        for q in range(n):
            gates.append(_gate("cz", [q, (q + 1) % n]))
            params.append(None)
    return gates, params


def _engine(gates):
    out = []
    for name, t, a, m in gates:
        if name == "unitary":
            out.append(G.Unitary(t, m))
        elif name in _FIXED:
            out.append(_CTOR[name](t))
        else:
            out.append(_CTOR[name](t, a))
    return out


def _chain(n, rng):
    """A rotated qubit entangled with the others in random order, between
    single-qubit rotations."""
    p = rng.permutation(n)
    out = [_gate("ry", [q], float(rng.uniform(0, 2 * math.pi))) for q in p[:n // 2]]
    return out + [_gate("cx", [p[0], q]) for q in p[1:]]


def _paulis(n, terms, rng):
    """Random weight-4 Pauli strings with normal coefficients."""
    w = min(4, n)
    return (["".join("XYZ"[int(i)] for i in rng.integers(0, 3, w)) for _ in range(terms)],
            [[int(q) for q in rng.choice(n, w, replace=False)] for _ in range(terms)],
            [float(c) for c in rng.standard_normal(terms)])


def _instances(case, rng):
    """MaxCut on random 3-regular simple graphs of even sizes."""
    sizes = list(range(case["lo"], case["hi"] + 1, 2))
    nq = [sizes[j % len(sizes)] for j in range(case["count"])]
    graphs = []
    for n in nq:
        while True:
            stubs = rng.permutation(np.repeat(np.arange(n), 3))
            e = {(int(min(a, b)), int(max(a, b))) for a, b in zip(stubs[::2], stubs[1::2]) if a != b}
            if len(e) == 3 * n // 2:
                break
        graphs.append(sorted(e))
    shape = (len(nq), case["p"])
    return nq, graphs, rng.uniform(0, math.pi, shape), rng.uniform(0, math.pi / 2, shape)


def _sizes(case):
    span = case["hi"] - case["lo"] + 1
    return [case["lo"] + j % span for j in range(case["count"])]


def _source(n, depth, rng):
    """OpenQASM 3 text of an ansatz-like circuit with rotations and CNOTs."""
    lines = ["OPENQASM 3.0;", f"qubit[{n}] q;"]
    gates = []
    for _ in range(depth):
        for q in range(n):
            for name in ("rx", "rz"):
                a = float(rng.uniform(0, 2 * math.pi))
                lines.append(f"{name}({a!r}) q[{q}];")
                gates.append(_gate(name, [q], a))
        p = rng.permutation(n)
        for w in range(n // 2):
            a, b = int(p[2 * w]), int(p[2 * w + 1])
            lines.append(f"cnot q[{a}], q[{b}];")
            gates.append(_gate("cx", [a, b]))
    lines += ["#pragma braket result state_vector", "#pragma braket result probability",
              f"#pragma braket result expectation z(q[0]) @ x(q[{n - 1}])"]
    return "\n".join(lines), gates


# --------------------------------------------------------------------------
# device buffers
# --------------------------------------------------------------------------
class _Amplitudes:
    """The array interface of a device state, for a torch view of it (the
    view holds this object, and this object the state's memory)."""

    def __init__(self, sv, dtype):
        self.sv = sv
        self.__cuda_array_interface__ = {
            "shape": (sv.num_elems(),), "typestr": "<c8" if dtype == "complex64" else "<c16",
            "data": (sv.data_ptr, False), "strides": None, "version": 2}


def _state(n, dtype):
    sv = _C.result_types.StateVector(_C.DeviceType.CUDA, n, dtype=dtype)
    F.initialize_basis_z(sv)
    return sv


def _view(sv, dtype):
    return torch.as_tensor(_Amplitudes(sv, dtype), device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = {"case": case}
    dt = case["dtype"]
    if kind == "gates":
        s["ops"] = _engine(_chain(case["n"], rng))
    elif kind == "program":
        ops = _engine(_circuit(case["style"], case["n"], case["depth"], rng))
        if case["fuse"]:
            ops = fuse_operations(ops, case["fuse"])
        s["program"] = F.Program(case["n"], ops, dtype=dt)
    elif kind == "adjoint":
        th = rng.uniform(0, 2 * math.pi, 2 * case["n"] * case["layers"])
        gates, params = _ansatz(case["n"], case["layers"], th)
        s["program"] = F.Program(case["n"], _engine(gates), dtype=dt)
        s["map"] = [[] if p is None else [(0, p)] for p in params]
        s["params"] = th.size
        s["obs"] = _paulis(case["n"], case["terms"], rng)
        s["work"] = [_state(case["n"], dt) for _ in range(3)]
        s["points"] = [_state(case["n"], dt) for _ in range(case["checkpoints"])]
    elif kind == "params":
        th = rng.uniform(0, 2 * math.pi, (case["sets"], 2 * case["n"] * case["layers"]))
        s["obs"] = _paulis(case["n"], case["terms"], rng)
        s["batch"] = ParameterBatch(
            case["n"], lambda t: _engine(_ansatz(case["n"], case["layers"], t)[0]), th, dtype=dt)
    elif kind == "circuits":
        circs = [(n, _engine(_circuit("layered", n, case["depth"], rng))) for n in _sizes(case)]
        s["batch"] = circuit_batch(circs, dtype=dt)
        s["states"] = [_state(n, dt) for n in _sizes(case)]
        s["views"] = [_view(sv, dt) for sv in s["states"]]
    elif kind == "qaoa":
        nq, graphs, s["gammas"], s["betas"] = _instances(case, rng)
        s["batch"] = qaoa_batch(nq, graphs, case["p"], dtype=dt)
    elif kind == "sample":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        v = torch.randn(1 << case["n"], 2, device="cuda", dtype=torch.float64, generator=gen)
        v /= v.norm()
        s["sv"] = _state(case["n"], dt)
        _view(s["sv"], dt).copy_(torch.view_as_complex(v))
        s["uniforms"] = rng.random(case["shots"])
    else:
        s["source"] = _source(case["n"], case["depth"], rng)[0]
        s["simulator"] = StateVectorSimulator()
    if kind in ("gates", "program"):
        s["sv"] = _state(case["n"], dt)
        s["view"] = _view(s["sv"], dt)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gates":
        F.initialize_basis_z(s["sv"])
        for op in s["ops"]:
            F.apply(s["sv"], op, case["n"], op.targets)
        return s["view"]
    if kind == "program":
        F.initialize_basis_z(s["sv"])
        s["program"].run(s["sv"], use_graph=case["graph"])
        return s["view"]
    if kind == "adjoint":
        e, grads = s["program"].adjoint(*s["work"], s["points"], s["map"], s["params"], *s["obs"])
        return {"energy": e, "grads": grads}
    if kind == "params":
        return s["batch"].energies(*s["obs"], use_graph=True)
    if kind == "circuits":
        s["batch"].run()
        for j, sv in enumerate(s["states"]):
            s["batch"].copy_state(j, sv)
        return s["views"]
    if kind == "qaoa":
        return s["batch"].run(s["gammas"], s["betas"])
    if kind == "sample":
        return F.sample(s["sv"], s["uniforms"], exact=True, normalize=case["dtype"] == "complex64")
    res = s["simulator"].run({"source": s["source"]}, shots=0, precision=case["dtype"])
    return [r["value"] if isinstance(r, dict) else r.value for r in res.resultTypes]


# --------------------------------------------------------------------------
# work of one pass: what it cannot do without
# --------------------------------------------------------------------------
def _gate_flops(gates, n):
    """Real operations of a gate list on one 2^n state (a dense matrix row is
    d complex products and d - 1 sums, a diagonal entry one product)."""
    f = 0.0
    for name, t, _, m in gates:
        d = 1 << len(t)
        nz = np.count_nonzero(m) / d
        moved = np.count_nonzero(~np.isclose(m, np.eye(d)).all(axis=1)) / d
        f += moved * (6 * nz + 2 * (nz - 1)) * 2.0 ** n
    return f


def work(case):
    kind = case["kind"]
    item = 8 if case["dtype"] == "complex64" else 16
    rng = np.random.default_rng(0)
    if kind == "gates":
        n = case["n"]
        return {"bytes": item * 2.0 ** n, "flops": _gate_flops(_chain(n, rng), n)}
    if kind == "program":
        n = case["n"]
        return {"bytes": item * 2.0 ** n,
                "flops": _gate_flops(_circuit(case["style"], n, case["depth"], rng), n)}
    if kind in ("adjoint", "params"):
        n, sets = case["n"], case.get("sets", 1)
        gates, _ = _ansatz(n, case["layers"], np.ones(2 * n * case["layers"]))
        f = sets * _gate_flops(gates, n)
        # each parameter set's state made once and read once by the strings
        # (8 operations an amplitude and string); the gradient undoes the
        # circuit on two states and takes one inner product a parameter
        f_obs = sets * case["terms"] * 8 * 2.0 ** n
        if kind == "adjoint":
            return {"bytes": 3 * item * 2.0 ** n,
                    "flops": 3 * f + f_obs + 2 * n * case["layers"] * 14 * 2.0 ** n}
        return {"bytes": 2 * item * sets * 2.0 ** n, "flops": f + f_obs}
    if kind == "circuits":
        f = sum(_gate_flops(_circuit("layered", n, case["depth"], rng), n) for n in _sizes(case))
        return {"bytes": 3.0 * item * sum(2.0 ** n for n in _sizes(case)), "flops": f}
    if kind == "qaoa":
        b = f = 0.0
        for n in _instances(case, rng)[0]:
            b += 2 * item * 2.0 ** n
            f += 3 * case["p"] * (6 + 8 * n) * 2.0 ** n
        return {"bytes": b, "flops": f}
    if kind == "sample":
        return {"bytes": item * 2.0 ** case["n"] + 16.0 * case["shots"],
                "flops": 4 * 2.0 ** case["n"]}
    n = case["n"]
    return {"bytes": (2 * item + 8) * 2.0 ** n,
            "flops": _gate_flops(_source(n, case["depth"], rng)[1], n)}


# --------------------------------------------------------------------------
# the same values in 64 bits, with torch alone
# --------------------------------------------------------------------------
def _zero(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1
    return psi


def _axes(psi, n, targets):
    """psi seen with one axis of 2 per target (ascending) and the rest
    between them, and the axis of each target."""
    ts = sorted(targets)
    shape, ax, last = [], {}, -1
    for t in ts:
        shape += [1 << (t - last - 1), 2]
        ax[t] = len(shape) - 1
        last = t
    shape.append(1 << (n - 1 - last))
    return psi.view(shape), [ax[t] for t in targets]


def _slices(v, ax):
    k = len(ax)
    out = []
    for r in range(1 << k):
        idx = [slice(None)] * v.dim()
        for j, a in enumerate(ax):
            idx[a] = (r >> (k - 1 - j)) & 1
        out.append(v[tuple(idx)])
    return out


def _apply(psi, n, targets, m):
    """In place: psi <- m on targets (targets[0] the most significant)."""
    v, ax = _axes(psi, n, targets)
    x = _slices(v, ax)
    d = len(x)
    rows = [r for r in range(d) if not (m[r, r] == 1 and np.count_nonzero(m[r]) == 1)]
    new = []
    for r in rows:
        y = None
        for c in range(d):
            if m[r, c] != 0:
                y = x[c] * complex(m[r, c]) if y is None else y.add_(x[c], alpha=complex(m[r, c]))
        new.append(y)
    for r, y in zip(rows, new):
        x[r].copy_(y)


def _evolve(n, gates):
    psi = _zero(n)
    for _, t, _, m in gates:
        _apply(psi, n, t, m)
    return psi


def _pauli_term(psi, n, pauli, qubits, idx):
    """P psi."""
    x = 0
    y = psi
    for p, q in zip(pauli, qubits):
        b = 1 << (n - 1 - q)
        if p in "XY":
            x |= b
    y = psi[idx ^ x] if x else psi.clone()
    sign = torch.zeros_like(idx)
    ny = 0
    for p, q in zip(pauli, qubits):
        if p in "YZ":
            sign ^= idx >> (n - 1 - q)
        ny += p == "Y"
    # Y = i X Z on the source bit, -i on the result's: (Y psi)_i = -i (-1)^b_i psi_(i^1) with b_i = 0
    y = y * (1 - 2 * (sign & 1)).to(torch.float64)
    return y * (-1j) ** ny


def _obs_apply(psi, n, obs):
    idx = torch.arange(psi.numel(), device=psi.device)
    out = torch.zeros_like(psi)
    for p, q, c in zip(*obs):
        out += c * _pauli_term(psi, n, p, q, idx)
    return out


def _exact_adjoint(case, rng):
    n = case["n"]
    th = rng.uniform(0, 2 * math.pi, 2 * n * case["layers"])
    gates, params = _ansatz(n, case["layers"], th)
    obs = _paulis(n, case["terms"], rng)
    psi = _evolve(n, gates)
    lam = _obs_apply(psi, n, obs)
    energy = float(torch.vdot(psi, lam).real)
    grads = torch.zeros(th.size, dtype=torch.float64, device="cuda")
    for (name, t, _, m), p in zip(reversed(gates), reversed(params)):
        if p is not None:
            # d/dtheta exp(-i theta P / 2) = -i/2 P exp(...): 2 Re <lam|dU|..> = Im <lam|P|psi>
            v, ax = _axes(psi, n, t)
            w, _ = _axes(lam, n, t)
            (v0, v1), (w0, w1) = _slices(v, ax), _slices(w, ax)
            if name == "rz":
                grads[p] = ((w0.conj() * v0).imag.sum() - (w1.conj() * v1).imag.sum())
            else:  # P = Y: (Y psi)_0 = -i psi_1, (Y psi)_1 = i psi_0
                grads[p] = ((w1.conj() * v0).real.sum() - (w0.conj() * v1).real.sum())
        inv = m.conj().T
        _apply(psi, n, t, inv)
        _apply(lam, n, t, inv)
    return {"energy": energy, "grads": grads.cpu()}


def _exact_params(case, rng):
    n = case["n"]
    th = torch.from_numpy(rng.uniform(0, 2 * math.pi, (case["sets"], 2 * n * case["layers"]))).cuda()
    obs = _paulis(n, case["terms"], rng)
    out = []
    for part in torch.split(th, 16):
        psi = torch.zeros(part.shape[0], 1 << n, dtype=torch.complex128, device="cuda")
        psi[:, 0] = 1
        c, s = torch.cos(part / 2), torch.sin(part / 2)
        p = 0
        for _ in range(case["layers"]):
            for name in ("ry", "rz"):
                for q in range(n):
                    v = psi.view(part.shape[0], 1 << q, 2, -1)
                    cc, ss = c[:, p, None, None], s[:, p, None, None]
                    x0, x1 = v[:, :, 0], v[:, :, 1]
                    if name == "ry":
                        y0, y1 = cc * x0 - ss * x1, ss * x0 + cc * x1
                    else:
                        ph = torch.complex(cc, ss)
                        y0, y1 = x0 * ph.conj(), x1 * ph
                    v[:, :, 0] = y0
                    v[:, :, 1] = y1
                    p += 1
            i = torch.arange(1 << n, device="cuda")
            par = torch.zeros_like(i)
            for q in range(n):
                par ^= (i >> (n - 1 - q)) & (i >> (n - 1 - (q + 1) % n))
            psi *= (1 - 2 * (par & 1)).to(torch.float64)
        for row in psi:
            out.append(float(torch.vdot(row, _obs_apply(row, n, obs)).real))
    return np.array(out)


def _exact_qaoa(case, rng):
    nq, graphs, gammas, betas = _instances(case, rng)
    out = np.empty((len(nq), 1 + 2 * case["p"]))
    for j, (n, edges) in enumerate(zip(nq, graphs)):
        i = torch.arange(1 << n, device="cuda")
        cut = torch.zeros(1 << n, dtype=torch.float64, device="cuda")
        for a, b in edges:
            cut += ((i >> (n - 1 - a)) ^ (i >> (n - 1 - b))) & 1
        spin = len(edges) - 2 * cut

        def mix(psi, beta):
            c, s = math.cos(beta), -1j * math.sin(beta)
            for q in range(n):
                v = psi.view(1 << q, 2, -1)
                x0 = v[:, 0].clone()
                v[:, 0].mul_(c).add_(v[:, 1], alpha=s)
                v[:, 1].mul_(c).add_(x0, alpha=s)

        psi = torch.full((1 << n,), 2.0 ** (-n / 2), dtype=torch.complex128, device="cuda")
        for g, b in zip(gammas[j], betas[j]):
            psi *= torch.exp(-1j * float(g) * spin)
            mix(psi, float(b))
        lam = cut * psi
        out[j, 0] = float(torch.vdot(psi, lam).real)
        for k in reversed(range(case["p"])):
            acc = 0.0
            for q in range(n):
                v, w = psi.view(1 << q, 2, -1), lam.view(1 << q, 2, -1)
                acc += float(((w[:, 0].conj() * v[:, 1]).sum() + (w[:, 1].conj() * v[:, 0]).sum()).imag)
            out[j, 1 + case["p"] + k] = 2 * acc
            mix(psi, -float(betas[j][k]))
            mix(lam, -float(betas[j][k]))
            out[j, 1 + k] = 2 * float((lam.conj() * psi * spin).sum().imag)
            ph = torch.exp(1j * float(gammas[j][k]) * spin)
            psi *= ph
            lam *= ph
    return out


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "gates":
        return _evolve(case["n"], _chain(case["n"], rng))
    if kind == "program":
        return _evolve(case["n"], _circuit(case["style"], case["n"], case["depth"], rng))
    if kind == "adjoint":
        return _exact_adjoint(case, rng)
    if kind == "params":
        return _exact_params(case, rng)
    if kind == "circuits":
        return [_evolve(n, _circuit("layered", n, case["depth"], rng)) for n in _sizes(case)]
    if kind == "qaoa":
        return _exact_qaoa(case, rng)
    if kind == "sample":
        return None  # whole numbers
    n = case["n"]
    psi = _evolve(n, _source(n, case["depth"], rng)[1])
    p = psi.real ** 2 + psi.imag ** 2
    x = psi.view(2, -1, 2)  # qubit 0 and qubit n - 1
    e = (x[0, :, 0].conj() * x[0, :, 1]).sum().real - (x[1, :, 0].conj() * x[1, :, 1]).sum().real
    return [psi, p, 2 * float(e)]
