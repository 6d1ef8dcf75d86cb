"""Programs whose gates run several to a pass (kernels_pass.hip): every chunk
size and the state sizes around it, against the CPU oracle."""
import ctypes
import os

import numpy as np
import pytest

from helpers import device_state, random_state, run_oracle, to_np

pytestmark = pytest.mark.gpu

# the bars of the gate tests: max-abs error of a unit-norm state
TOL = {"complex128": 1e-12, "complex64": 1e-5}


def _circuit(n, rng, gates):
    """Random gates of 0-5 targets: all kinds, dense blocks of 4 and 5 targets
    on random qubits, global phases, controls."""
    from snuqs_amd.circuits import haar_unitary, random_gate_list
    from snuqs_amd._C.operation import gate_operations as g

    ops = []
    for op in random_gate_list(n, gates, rng, with_unitary=True):
        ops.append(op)
        if rng.random() < 0.15:
            k = int(rng.integers(4, 6))
            ops.append(g.Unitary([int(q) for q in rng.permutation(n)[:k]], haar_unitary(1 << k, rng)))
    return ops + [g.RotX([int(q) for q in rng.permutation(n)[:3]], 0.7, ctrl_modifiers=[1, 0]),
                  g.GPhase([], 0.9)]


# 8 / 9: below the smallest chunk of complex128 / complex64; 9-13: the state is
# one chunk; 20 / 21: the largest chunk starts at 20 (complex64) and 21 qubits
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [8, 9, 10, 11, 12, 13, 14, 17, 20, 21])
def test_program_passes_vs_oracle(C, dtype, n):
    rng = np.random.default_rng(1000 + n)
    ops = _circuit(n, rng, 60)
    init = random_state(n, rng, np.complex64 if dtype == "complex64" else np.complex128)
    ref = run_oracle(n, ops, init.astype(np.complex128))
    prog = C.functionals.Program(n, ops, dtype=dtype)
    for use_graph in (False, True):
        sv = device_state(C, n, dtype, init)
        prog.run(sv, use_graph=use_graph)
        assert np.abs(to_np(C, sv) - ref).max() <= TOL[dtype], use_graph


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_set_gates_from_identities(C, dtype):
    """A program made with all angles 0 (every gate the identity) runs the
    gates that later matrices make of it."""
    from snuqs_amd.circuits import hea_ansatz

    n = 14
    th = np.random.default_rng(4).uniform(0, 2 * np.pi, 4 * n)
    prog = C.functionals.Program(n, hea_ansatz(n, 2, 0 * th)[0], dtype=dtype)
    ops = hea_ansatz(n, 2, th)[0]
    prog.set_gates(ops)
    sv = device_state(C, n, dtype)
    prog.run(sv)
    assert np.abs(to_np(C, sv) - run_oracle(n, ops)).max() <= TOL[dtype]


P = ctypes.c_void_p


def _library(C):
    L = ctypes.CDLL(os.path.join(os.path.dirname(C.__file__), "libsnuqs_hip.so"))
    U32 = ctypes.c_uint32
    L.sq_memcpy_h2d.argtypes = [P, P, ctypes.c_size_t, P]
    L.sq_program_create.argtypes = [ctypes.POINTER(P), ctypes.c_int, U32, U32, P, P, P]
    L.sq_program_run.argtypes = [P, P, ctypes.c_uint64, P]
    L.sq_program_destroy.argtypes = [P]
    L.sq_batch_create.argtypes = [ctypes.POINTER(P), ctypes.c_int, U32, U32, U32, P, P, P]
    L.sq_batch_run.argtypes = [P, P, ctypes.c_uint64, P]
    L.sq_batch_run_graph.argtypes = [P, P, ctypes.c_uint64, P]
    L.sq_batch_destroy.argtypes = [P]
    return L


def _rotations(C, n, th):
    """Gates that are the identity at angle 0."""
    g = C.operation.gate_operations
    ops = [g.RotX([q], float(th[q])) for q in range(n)]
    ops += [g.XX([q, q + 1], float(th[n + q])) for q in range(n - 1)]
    return ops + [g.RotZ([q], float(th[q] * th[n - 1 - q])) for q in range(n)]


# rounding tells a plan from another, so equal bits are equal steps
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_steps_follow_the_matrices(C, dtype):
    """A program's steps are those of a program made with its present matrices,
    whatever it was made with (angles of 0 and others)."""
    n = 12
    th = [np.zeros(2 * n)] + list(np.random.default_rng(5).uniform(0.1, 3, (2, 2 * n)))
    fresh = []
    for t in th:
        sv = device_state(C, n, dtype)
        C.functionals.Program(n, _rotations(C, n, t), dtype=dtype).run(sv)
        fresh.append(to_np(C, sv))
    for order in ((0, 1, 2), (1, 0, 2, 1)):
        prog = C.functionals.Program(n, _rotations(C, n, th[order[0]]), dtype=dtype)
        for i in order:
            prog.set_gates(_rotations(C, n, th[i]))
            for use_graph in (False, True):
                sv = device_state(C, n, dtype)
                prog.run(sv, use_graph=use_graph)
                assert np.array_equal(to_np(C, sv), fresh[i]), (order, i, use_graph)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_batch_steps_follow_the_matrices(C, dtype):
    from snuqs_amd.batch import BatchProgram, StateBatch

    n, sets = 12, 3
    rng = np.random.default_rng(6)
    zero = np.zeros((sets, 2 * n))
    some = rng.uniform(0.1, 3, (sets, 2 * n))
    mixed = some * (np.arange(sets) % 2)[:, None]  # set 0 (and 2) at zero beside another
    states = StateBatch(sets, n, dtype=dtype)

    def run(b, use_graph=False):
        states.initialize_basis_z()
        b.run(states, use_graph=use_graph)
        return np.array(states.cpu(), copy=True)

    def circuits(th):
        return [_rotations(C, n, t) for t in th]

    fresh = {name: run(BatchProgram(n, circuits(th), dtype=dtype))
             for name, th in (("zero", zero), ("some", some), ("mixed", mixed))}
    th = {"zero": zero, "some": some, "mixed": mixed}
    b = BatchProgram(n, circuits(zero), dtype=dtype)
    for name in ("some", "zero", "mixed", "zero", "some"):
        b.set_gates(circuits(th[name]))
        for use_graph in (False, True):
            assert np.array_equal(run(b, use_graph), fresh[name]), (name, use_graph)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_new_matrices_then_a_callers_capture(C, dtype):
    """The first run after set_gates inside a graph that the caller captures,
    and later runs on two streams at once."""
    import threading

    n = 14
    th = np.random.default_rng(9).uniform(0, 3, (2, 2 * n))
    prog = C.functionals.Program(n, _rotations(C, n, th[0]), dtype=dtype)
    ref = run_oracle(n, _rotations(C, n, th[1]))
    sv = device_state(C, n, dtype)
    prog.run(sv)
    prog.set_gates(_rotations(C, n, th[1]))
    L = _library(C)  # (finds the HIP runtime that the engine runs on)
    L.hipStreamBeginCapture.argtypes = [P, ctypes.c_int]
    L.hipStreamEndCapture.argtypes = [P, ctypes.POINTER(P)]
    L.hipGraphInstantiate.argtypes = [ctypes.POINTER(P), P, P, P, ctypes.c_size_t]
    L.hipGraphLaunch.argtypes = [P, P]
    L.hipGraphExecDestroy.argtypes = L.hipGraphDestroy.argtypes = [P]
    stream = C.stream.Stream.create_nonblocking()
    graph, executable = P(), P()
    C.core.cuda.device_synchronize()
    assert L.hipStreamBeginCapture(stream.get(), 0) == 0  # global mode
    C.functionals.initialize_basis_z(sv, stream=stream)
    prog.run(sv, stream=stream)
    assert L.hipStreamEndCapture(stream.get(), ctypes.byref(graph)) == 0
    assert L.hipGraphInstantiate(ctypes.byref(executable), graph, None, None, 0) == 0
    for _ in range(3):
        assert L.hipGraphLaunch(executable, stream.get()) == 0
        C.core.cuda.device_synchronize()
        assert np.abs(to_np(C, sv) - ref).max() <= TOL[dtype]
        C.functionals.norm2(sv)
    L.hipGraphExecDestroy(executable)
    L.hipGraphDestroy(graph)
    # eager again, from two threads at once
    svs = [device_state(C, n, dtype) for _ in range(2)]
    C.core.cuda.device_synchronize()
    streams = [C.stream.Stream.create() for _ in svs]
    threads = [threading.Thread(target=prog.run, args=(s,), kwargs={"stream": st})
               for s, st in zip(svs, streams)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    C.core.cuda.device_synchronize()
    fresh = device_state(C, n, dtype)
    C.functionals.Program(n, _rotations(C, n, th[1]), dtype=dtype).run(fresh)
    for s in svs:
        assert np.array_equal(to_np(C, s), to_np(C, fresh))


def _gate_arrays(ops):
    return (np.array([len(op.targets) for op in ops], np.uint32),
            np.array([q for op in ops for q in op.targets], np.uint32),
            np.concatenate([np.asarray(op.matrix(), np.complex128).ravel() for op in ops]))


def test_unaligned_complex64_state(C):
    """A complex64 state at an odd amplitude (8 bytes past a 16-byte
    boundary), as a C caller may hold it, gets the same result."""
    L = _library(C)
    n = 14
    rng = np.random.default_rng(6)
    ops = _circuit(n, rng, 30)
    init = random_state(n, rng, np.complex64)
    buf = C.result_types.StateVector(C.DeviceType.CUDA, n + 1, dtype="complex64")
    host = np.zeros(2 << n, np.complex64)
    host[1:1 + (1 << n)] = init
    nt, tg, ms = _gate_arrays(ops)
    prog = P()
    assert L.sq_memcpy_h2d(buf.data_ptr, host.ctypes.data, host.nbytes, None) == 0
    assert L.sq_program_create(ctypes.byref(prog), 0, n, len(ops), nt.ctypes.data, tg.ctypes.data,
                               ms.ctypes.data) == 0
    assert L.sq_program_run(prog, buf.data_ptr + 8, 1 << n, None) == 0
    C.core.cuda.device_synchronize()
    out = np.array(buf.cpu(), copy=True)
    L.sq_program_destroy(prog)
    got = out[1:1 + (1 << n)].astype(np.complex128)
    assert np.abs(got - run_oracle(n, ops, init.astype(np.complex128))).max() <= TOL["complex64"]
    assert out[0] == 0 and not out[1 + (1 << n):].any()  # nothing beside the state


@pytest.mark.parametrize("dtype,at", [("complex64", 8), ("complex128", 16)])
def test_unaligned_batch_states(C, dtype, at):
    """The states of a parameter batch one element past the buffer's start."""
    L = _library(C)
    n, sets = 12, 3
    rng = np.random.default_rng(7)
    circuits = [_circuit(n, np.random.default_rng(8), 30) for _ in range(sets)]
    nt, tg, _ = _gate_arrays(circuits[0])
    ms = np.concatenate([_gate_arrays(ops)[2] for ops in circuits])
    init = [random_state(n, rng, np.dtype(dtype)) for _ in range(sets)]
    batch = P()
    assert L.sq_batch_create(ctypes.byref(batch), dtype == "complex128", n, sets, len(nt),
                             nt.ctypes.data, tg.ctypes.data, ms.ctypes.data) == 0
    buf = C.result_types.StateVector(C.DeviceType.CUDA, n + 2, dtype=dtype)
    for run in (L.sq_batch_run, L.sq_batch_run_graph):
        host = np.zeros(4 << n, dtype)
        host[1:1 + (sets << n)] = np.concatenate(init)
        assert L.sq_memcpy_h2d(buf.data_ptr, host.ctypes.data, host.nbytes, None) == 0
        assert run(batch, buf.data_ptr + at, 1 << n, None) == 0
        C.core.cuda.device_synchronize()
        out = np.array(buf.cpu(), copy=True)
        for y in range(sets):
            got = out[1 + (y << n):1 + ((y + 1) << n)].astype(np.complex128)
            ref = run_oracle(n, circuits[y], init[y].astype(np.complex128))
            assert np.abs(got - ref).max() <= TOL[dtype], y
        assert out[0] == 0 and not out[1 + (sets << n):].any()
    L.sq_batch_destroy(batch)


# 64 MiB: the smallest state above 2 MiB that passes read with ordinary accesses
@pytest.mark.parametrize("dtype,n", [("complex128", 22), ("complex64", 23)])
def test_passes_with_ordinary_accesses(C, dtype, n):
    rng = np.random.default_rng(n)
    ops = _circuit(n, rng, 12)
    init = random_state(n, rng, np.complex64 if dtype == "complex64" else np.complex128)
    sv = device_state(C, n, dtype, init)
    C.functionals.Program(n, ops, dtype=dtype).run(sv)
    assert np.abs(to_np(C, sv) - run_oracle(n, ops, init.astype(np.complex128))).max() <= TOL[dtype]


# 32 MiB: the smallest state that single gates read with ordinary accesses; a
# diagonal, a swap, dense gates of 1 to 5 targets, low, high and mixed bits
@pytest.mark.parametrize("dtype,n", [("complex128", 21), ("complex64", 22)])
def test_gates_with_ordinary_accesses(C, dtype, n):
    from snuqs_amd.circuits import haar_unitary
    from snuqs_amd._C.operation import gate_operations as g

    rng = np.random.default_rng(n)
    ops = [g.Hadamard([0]), g.Hadamard([n - 1]), g.RotZ([3], 0.4), g.CX([1, n - 2]),
           g.Swap([0, n - 1]), g.CCNot([2, n // 2, n - 1])]
    for k in (2, 3, 4, 5):
        for t in (list(range(k)), list(range(n - k, n)), [int(q) for q in rng.permutation(n)[:k]]):
            ops.append(g.Unitary(t, haar_unitary(1 << k, rng)))
    init = random_state(n, rng, np.complex64 if dtype == "complex64" else np.complex128)
    sv = device_state(C, n, dtype, init)
    for op in ops:
        C.functionals.apply(sv, op, n, op.targets)
    assert np.abs(to_np(C, sv) - run_oracle(n, ops, init.astype(np.complex128))).max() <= TOL[dtype]


# 512 MiB: gates that touch half of it or less are read with ordinary accesses,
# full sweeps are not
@pytest.mark.parametrize("dtype,n", [("complex128", 25), ("complex64", 26)])
def test_gates_on_a_state_beyond_the_caches(C, dtype, n):
    from snuqs_amd._C.operation import gate_operations as g

    small = 6  # the same gates on the qubits that they touch
    where = [0, 3, 10, n - 9, n - 2, n - 1]
    rng = np.random.default_rng(n)
    gates = [lambda q: g.RotY(q[:1], 0.7), lambda q: g.CX(q[:2]), lambda q: g.CZ(q[:2]),
             lambda q: g.RotZ(q[:1], 0.3), lambda q: g.Swap(q[:2]), lambda q: g.CCNot(q[:3])]
    sv = device_state(C, n, dtype)
    ops = []
    for i in range(36):
        q = [int(x) for x in rng.permutation(small)]
        ops.append(gates[i % 6](q))
        op = gates[i % 6]([where[x] for x in q])
        C.functionals.apply(sv, op, n, op.targets)
    ref = run_oracle(small, ops)
    index = [sum(((i >> (small - 1 - j)) & 1) << (n - 1 - where[j]) for j in range(small))
             for i in range(1 << small)]
    got = np.array(C.functionals.amplitudes(sv, index))
    assert np.abs(got - ref).max() <= TOL[dtype]
    assert abs(C.functionals.norm2(sv) - 1) <= TOL[dtype]


@pytest.fixture
def little_memory(C):
    """take(mib): device memory taken until that many MiB or less are left."""
    L = _library(C)
    L.sq_malloc.argtypes = [ctypes.POINTER(P), ctypes.c_size_t]
    L.sq_free.argtypes = [P]
    held = []

    def take(mib):
        left = mib << 20
        size = C.core.cuda.mem_info()[0] - left
        while size >= 1 << 20:
            p = P()
            if L.sq_malloc(ctypes.byref(p), size) == 0:
                held.append(p)
                size = min(size, C.core.cuda.mem_info()[0] - left)
            else:
                size //= 2
        assert C.core.cuda.mem_info()[0] <= left + (4 << 20)

    yield take
    for p in held:
        L.sq_free(p)


def _small_gates(n, gates, seed):
    from snuqs_amd.circuits import haar_unitary
    from snuqs_amd._C.operation import gate_operations as g

    where, rng = np.random.default_rng(n), np.random.default_rng(seed)
    return [g.Unitary([int(q) for q in where.permutation(n)[:k]], haar_unitary(1 << k, rng))
            for k in where.integers(1, 3, gates)]


def test_program_without_room_for_passes(C, little_memory):
    """60,000 gates on 10 qubits: some 100 MB of pass matrices."""
    n = 10
    ops = _small_gates(n, 60000, 1)
    sv = device_state(C, n, "complex128")
    little_memory(64)
    prog = C.functionals.Program(n, ops, dtype="complex128")
    prog.run(sv)
    # 60,000 roundings of 2^-53 on a unit vector, in the same order as the oracle
    assert np.abs(to_np(C, sv) - run_oracle(n, ops)).max() <= 1e-11


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_batch_without_room_for_passes(C, little_memory, dtype):
    """2,048 sets of 120 gates on 10 qubits: 6 KiB or more a block and set,
    some 250 MB, where the gates' own tables are 20; new matrices too."""
    from snuqs_amd.batch import BatchProgram, StateBatch

    n, sets, gates = 10, 2048, 120
    different = [_small_gates(n, gates, seed) for seed in range(3)]
    states = StateBatch(sets, n, dtype=dtype)
    little_memory(64)
    b = BatchProgram(n, [different[y % 3] for y in range(sets)], dtype=dtype)
    for first in (0, 1):
        if first:
            b.set_gates([different[(y + 1) % 3] for y in range(sets)])
        for use_graph in (False, True):
            states.initialize_basis_z()
            b.run(states, use_graph=use_graph)
            for y in (0, 1, 2, sets - 1):
                got = np.array(states.state(y).cpu(), copy=True).astype(np.complex128)
                ref = run_oracle(n, different[(y + first) % 3])
                assert np.abs(got - ref).max() <= TOL[dtype], (y, use_graph)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_circuit_batch_without_room_for_passes(C, little_memory, dtype):
    """2,048 circuits of 120 gates on 10 qubits: some 300 MB of pass matrices,
    where the states, matrices and tables are 75 to 115."""
    from snuqs_amd.cbatch import circuit_batch

    n, circuits, gates = 10, 2048, 120
    different = [_small_gates(n, gates, seed) for seed in range(3)]
    little_memory(160)
    b = circuit_batch([(n, different[y % 3]) for y in range(circuits)], dtype=dtype, fuse=False)
    for use_graph in (False, True):
        b.run(use_graph=use_graph)
        for y in (0, 1, 2, circuits - 1):
            got = b.state(y).astype(np.complex128)
            assert np.abs(got - run_oracle(n, different[y % 3])).max() <= TOL[dtype], (y, use_graph)


def _phases_and_permutations(C, n, rng, gates=25):
    """Gates that move and turn amplitudes without mixing them."""
    g = C.operation.gate_operations
    ops = []
    for _ in range(gates):
        q = [int(x) for x in rng.permutation(n)[:3]]
        a = float(rng.uniform(0.1, 3))
        ops.append([lambda: g.PauliX(q[:1]), lambda: g.S(q[:1]), lambda: g.T(q[:1]),
                    lambda: g.RotZ(q[:1], a), lambda: g.CX(q[:2]), lambda: g.CPhaseShift(q[:2], a),
                    lambda: g.Swap(q[:2]), lambda: g.ISwap(q[:2]), lambda: g.ZZ(q[:2], a),
                    lambda: g.CCNot(q)][int(rng.integers(10))]())
    return ops


# every chunk size of both types
@pytest.mark.parametrize("dtype,n", [("complex64", 10), ("complex64", 11), ("complex64", 14),
                                     ("complex64", 20), ("complex128", 9), ("complex128", 10),
                                     ("complex128", 14), ("complex128", 21)])
def test_large_amplitudes(C, dtype, n):
    """Amplitudes up to bf16's largest value (complex64) and to the largest
    double (blocks of 4 targets) keep their values beside ordinary ones."""
    rng = np.random.default_rng(n)
    ops = _phases_and_permutations(C, n, rng)
    init = random_state(n, rng, np.dtype(dtype))
    init[rng.permutation(1 << n)[:4]] = np.array([1, -1, 1j, -1j]) * (
        3.38e38 if dtype == "complex64" else 1.7e308)
    alone = device_state(C, n, dtype, init)
    for op in ops:
        C.functionals.apply(alone, op, n, op.targets)
    together = device_state(C, n, dtype, init)
    C.functionals.Program(n, ops, dtype=dtype).run(together)
    got, ref = to_np(C, together) * 2.0 ** -10, to_np(C, alone) * 2.0 ** -10
    # 25 products of an amplitude with a number of modulus 1
    tol = (1e-5 if dtype == "complex64" else 1e-13) * np.abs(ref).clip(2.0 ** (-n / 2 - 10))
    assert (np.abs(got - ref) <= tol).all()


def test_small_complex64_amplitudes(C):
    """The three bf16 parts of an amplitude hold its 24 bits down to 2^-108."""
    n = 12
    rng = np.random.default_rng(n)
    ops = _small_gates(n, 20, 3)
    init = (random_state(n, rng) * 2.0 ** -100).astype(np.complex64)  # 2^-106 each
    sv = device_state(C, n, "complex64", init)
    C.functionals.Program(n, ops, dtype="complex64").run(sv)
    ref = run_oracle(n, ops, init.astype(np.complex128))
    # 20 roundings of 2^-24, as at any other scale
    assert np.linalg.norm(to_np(C, sv) - ref) <= 20 * 2.0 ** -24 * np.linalg.norm(ref)
