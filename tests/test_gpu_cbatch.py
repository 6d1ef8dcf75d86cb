"""Circuits of uneven qubit counts as one launch sequence (sq_cbatch_*):
every circuit's state against the FP64 CPU oracle and against the same
circuit run alone as a Program; graph replays against eager runs; the
largest offsets (a 26-qubit circuit beside small ones); copy_state's checks."""
import numpy as np
import pytest

from helpers import device_state, run_oracle, to_np

pytestmark = pytest.mark.gpu


def _mixed_circuit(C, n, rng, depth):
    """Gates of 1-3 targets of every kind (dense, diagonal, permutation,
    controlled) plus 4-5 target blocks once fused."""
    from snuqs_amd.circuits import random_layered

    g = C.operation.gate_operations
    ops = [g.Hadamard([q]) for q in range(n)]
    if n >= 2:
        ops += random_layered(n, depth, seed=int(rng.integers(1 << 30)))
        ops += [g.CX([0, n - 1]), g.RotZ([n - 1], 0.3), g.Swap([0, 1])]
    if n >= 3:
        ops += [g.RotX([2, 0, 1], 0.7, ctrl_modifiers=[1, 0]), g.CCNot([1, 2, 0])]
    ops += [g.RotY([q], float(rng.uniform(0, 6.28))) for q in range(n)]
    return ops


@pytest.mark.parametrize("dtype,tol", [("complex128", 1e-12), ("complex64", 2e-5)])
@pytest.mark.parametrize("fuse", [False, True])
def test_cbatch_vs_oracle_and_programs(C, dtype, tol, fuse):
    from snuqs_amd.cbatch import circuit_batch
    from snuqs_amd.transpile import fuse_operations

    rng = np.random.default_rng(5)
    sizes = [3, 10, 1, 12, 7, 9, 2, 11]
    circs = [(n, _mixed_circuit(C, n, rng, 3)) for n in sizes]
    batch = circuit_batch(circs, dtype=dtype, fuse=fuse)
    batch.run(use_graph=False)
    st = batch.stats()
    nblocks = {n: len(fuse_operations(ops, 5)) if fuse else len(ops) for n, ops in circs}
    # one launch a step for the circuits below 10 / 9 qubits, and one a step and
    # chunk size (the qubit counts from there to 12 / 11) for the others' passes
    least = 10 if dtype == "complex64" else 9
    alone = max(b for n, b in nblocks.items() if n < least)
    chunks = len({min(n, least + 2) for n in sizes if n >= least})
    passes = max(b for n, b in nblocks.items() if n >= least)
    assert 2 + alone + chunks <= st["launches"] <= 2 + alone + chunks * passes
    for j, (n, ops) in enumerate(circs):
        got = batch.state(j).astype(np.complex128)
        ref = run_oracle(n, ops)
        assert np.abs(got - ref).max() < tol, (j, n)
        # the same blocks run alone through a Program
        prog_ops = fuse_operations(ops, 5) if fuse else ops
        sv = device_state(C, n, dtype)
        C.functionals.Program(n, prog_ops, dtype=dtype).run(sv)
        assert np.abs(got - to_np(C, sv)).max() < tol, (j, n)


def test_cbatch_graph_replays_match_eager(C):
    from snuqs_amd.cbatch import circuit_batch
    from snuqs_amd.circuits import random_layered

    circs = [(n, random_layered(n, 4, seed=n)) for n in (14, 6, 18, 13, 16)]
    batch = circuit_batch(circs, dtype="complex64")
    batch.run(use_graph=False)
    eager = [batch.state(j) for j in range(len(circs))]
    for r in range(3):
        batch.run(use_graph=True)  # captured on the first call, replayed after
        C.core.cuda.device_synchronize()
        for j in range(len(circs)):
            assert np.array_equal(batch.state(j), eager[j]), (r, j)


def test_cbatch_uneven_gate_counts_and_large_offsets(C):
    """A 26-qubit circuit (its state past 2^28 bytes of offsets for the ones
    after it) beside circuits of 0, 1 and many blocks; complex128 against
    Programs run alone (the oracle for the small ones)."""
    from snuqs_amd.cbatch import circuit_batch
    from snuqs_amd.circuits import random_layered
    from snuqs_amd.transpile import fuse_operations

    g = C.operation.gate_operations
    circs = [(5, []), (4, [g.Hadamard([2])]), (26, random_layered(26, 3, seed=2)),
             (8, random_layered(8, 12, seed=3)), (20, random_layered(20, 2, seed=4))]
    batch = circuit_batch(circs, dtype="complex128")
    batch.run()
    for j, (n, ops) in enumerate(circs):
        got = batch.state(j)
        if n <= 12:
            ref = run_oracle(n, ops)
        else:
            sv = device_state(C, n, "complex128")
            C.functionals.Program(n, fuse_operations(ops, 5), dtype="complex128").run(sv)
            ref = to_np(C, sv)
        assert np.abs(got - ref).max() < 1e-12, (j, n)
        assert abs(np.vdot(got, got).real - 1.0) < 1e-12, (j, n)


def test_cbatch_more_chunks_than_one_launch(C):
    """32 circuits of 30 qubits between two of 20 (256 GiB): 2^22 + 256 chunks
    in a step, more than one launch holds."""
    from snuqs_amd.cbatch import circuit_batch

    if C.core.cuda.mem_info()[0] < (257 << 30):
        pytest.skip("needs 257 GiB of free device memory")
    g = C.operation.gate_operations
    small = [g.RotY([3], 0.4), g.Hadamard([19])]
    batch = circuit_batch([(20, small)] + [(30, [g.Hadamard([5])])] * 32 + [(20, small)],
                          dtype="complex64", fuse=False)
    batch.run(use_graph=False)
    ref = run_oracle(20, small)
    for j in (0, 33):
        assert np.abs(batch.state(j).astype(np.complex128) - ref).max() < 1e-6, j


def test_cbatch_copy_state_checks(C):
    from snuqs_amd.cbatch import circuit_batch

    g = C.operation.gate_operations
    batch = circuit_batch([(3, [g.Hadamard([0])]), (5, [g.CX([0, 4])])], dtype="complex64")
    batch.run()
    with pytest.raises(ValueError):  # wrong size
        batch.copy_state(0, C.result_types.StateVector(C.DeviceType.CUDA, 5, dtype="complex64"))
    with pytest.raises(ValueError):  # wrong dtype
        batch.copy_state(1, C.result_types.StateVector(C.DeviceType.CUDA, 5, dtype="complex128"))
    with pytest.raises(IndexError):
        batch.copy_state(2, C.result_types.StateVector(C.DeviceType.CUDA, 5, dtype="complex64"))
    sv = C.result_types.StateVector(C.DeviceType.CUDA, 5, dtype="complex64")
    batch.copy_state(1, sv)
    a = np.array(sv.cpu())
    assert a[0] == 1 and np.count_nonzero(a) == 1


@pytest.mark.parametrize("dtype,tol", [("complex64", 2e-5), ("complex128", 1e-12)])
def test_cbatch_many_circuits(C, dtype, tol):
    """300 circuits (more entries per launch than a workgroup stages in LDS,
    so entries are found by the global search), 2-11 qubits, fused (5-target
    blocks on states with full tiles take the MFMA entry table) against the
    oracle; a second run of the batch gives the same bits."""
    from snuqs_amd.cbatch import circuit_batch
    from snuqs_amd.circuits import random_layered

    rng = np.random.default_rng(300)
    sizes = [int(rng.integers(2, 12)) for _ in range(300)]
    circs = [(n, random_layered(n, 3, seed=5000 + j)) for j, n in enumerate(sizes)]
    batch = circuit_batch(circs, dtype=dtype)
    batch.run()
    picks = [int(j) for j in rng.choice(len(circs), 40, replace=False)]
    first = {j: batch.state(j) for j in picks}
    for j in picks:
        n, ops = circs[j]
        got = first[j].astype(np.complex128)
        assert np.abs(got - run_oracle(n, ops)).max() < tol, (j, n)
    batch.run()
    for j in picks:
        assert np.array_equal(batch.state(j), first[j]), j


@pytest.mark.parametrize("dtype,sizes,launches", [
    # below the smallest chunk; every chunk size (2^13 amplitudes of complex64
    # from 2^20 in all, 2^12 of complex128 from 2^21); two circuits of one size;
    # no gates
    ("complex64", [8, 10, 11, 12, 13, 20, 3, 11], 2 + 1 + 4),
    ("complex128", [8, 9, 10, 11, 12, 21, 3, 10], 2 + 1 + 4),
    # passes only: nothing to zero
    ("complex64", [12, 12, 14], 1), ("complex128", [11, 13], 1)])
def test_cbatch_chunk_sizes(C, dtype, sizes, launches):
    """One batch of circuits of every chunk size: launches and bytes of a run
    of one gate each, and the states of longer circuits against the oracle."""
    from snuqs_amd.cbatch import circuit_batch
    from snuqs_amd.circuits import random_layered

    g = C.operation.gate_operations
    item = 8 if dtype == "complex64" else 16
    least = 10 if dtype == "complex64" else 9
    one = [(n, [] if n == 3 else [g.RotX([n - 2], 0.3)]) for n in sizes]
    batch = circuit_batch(one, dtype=dtype)
    batch.run()
    st = batch.stats()
    assert st["launches"] == launches
    amps = sum(1 << n for n in sizes)
    zeroed = amps if min(sizes) < least else 0
    # a first pass writes its state, a gate alone reads and writes it
    moved = sum((0 if n == 3 else 2 if n < least else 1) << n for n in sizes)
    assert st["traffic_bytes"] == item * (zeroed + moved)
    deep = [(n, [] if n == 3 else random_layered(n, 3, seed=40 + j)) for j, n in enumerate(sizes)]
    tol = 2e-5 if dtype == "complex64" else 1e-12
    for circs in (one, deep):
        batch = circuit_batch(circs, dtype=dtype)
        batch.run()
        for j, (n, ops) in enumerate(circs):
            got = batch.state(j).astype(np.complex128)
            assert np.abs(got - run_oracle(n, ops)).max() < tol, (j, n)


def test_cbatch_of_large_circuits(C):
    """40 circuits of 20 qubits agree with Programs run alone."""
    from snuqs_amd.cbatch import circuit_batch
    from snuqs_amd.circuits import random_layered
    from snuqs_amd.transpile import fuse_operations

    circs = [(20, random_layered(20, 3, seed=700 + j)) for j in range(40)]
    batch = circuit_batch(circs, dtype="complex64")
    batch.run()
    for j in (0, 13, 39):
        sv = device_state(C, 20, "complex64")
        C.functionals.Program(20, fuse_operations(circs[j][1], 5), dtype="complex64").run(sv)
        assert np.abs(batch.state(j).astype(np.complex128) - to_np(C, sv)).max() < 2e-5, j
