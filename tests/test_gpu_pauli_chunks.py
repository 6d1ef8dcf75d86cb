"""Expectations whose terms are formed several to a read of the state
(k_pauli_chunk): values against numpy, the sizes where chunks start, strings
of every weight, more terms than one launch, batches against single states."""
import numpy as np
import pytest

from helpers import device_state, random_state

pytestmark = pytest.mark.gpu


def _terms(n, rng):
    """Diagonal strings, weights 1-4, strings longer than a chunk holds, and
    several with the same mask; 150 in all (three launches)."""
    paulis, qubits = [], []
    for t in range(150):
        w = int(rng.integers(1, 5)) if t % 10 else int(rng.integers(1, n + 1))
        p = "".join("XYZ"[int(i)] for i in rng.integers(0, 3, w))
        if t % 7 == 3:
            p = "Z" * w
        paulis.append(p)
        qubits.append([int(q) for q in rng.choice(n, w, replace=False)])
    paulis += ["X" * n, "Y" * n, "Z" * n]
    qubits += [list(range(n))] * 3
    return paulis, qubits, [float(c) for c in rng.standard_normal(len(paulis))]


def _value(v, n, pauli, qubits, idx):
    x = z = 0
    for p, q in zip(pauli, qubits):
        b = 1 << (n - 1 - q)
        x |= b if p in "XY" else 0
        z |= b if p in "YZ" else 0
    sign = 1.0 - 2.0 * (np.bitwise_count(idx & z) & 1)
    # <v|P|v> = sum_i conj(v_{i^x}) i^ny (-1)^{|i & z|} v_i
    return float(np.real((1j) ** pauli.count("Y") * np.sum(np.conj(v[idx ^ x]) * sign * v)))


@pytest.mark.parametrize("dtype,n", [("complex64", 19), ("complex64", 20), ("complex64", 21),
                                     ("complex128", 18), ("complex128", 19), ("complex128", 20)])
def test_expectation_chunks(C, dtype, n):
    rng = np.random.default_rng(n)
    v = random_state(n, rng, np.complex64 if dtype == "complex64" else np.complex128)
    sv = device_state(C, n, dtype, v)
    paulis, qubits, coeffs = _terms(n, rng)
    e, terms = C.functionals.expectation(sv, paulis, qubits, coeffs)
    v = v.astype(np.complex128)
    idx = np.arange(1 << n)
    ref = np.array([_value(v, n, p, q, idx) for p, q in zip(paulis, qubits)])
    # both sides sum products of the same amplitudes in FP64: 2^n terms below
    # 2^-n each, errors far below n eps
    assert np.abs(np.asarray(terms) - ref).max() < 1e-13
    assert abs(e - float(np.dot(coeffs, ref))) < 1e-12


@pytest.mark.parametrize("dtype,n", [("complex64", 20), ("complex128", 19)])
def test_batch_values_are_the_states_values(C, dtype, n):
    from snuqs_amd.batch import ParameterBatch
    from snuqs_amd.circuits import hea_ansatz

    rng = np.random.default_rng(3)
    th = rng.uniform(0, 2 * np.pi, (3, 2 * n))
    b = ParameterBatch(n, lambda t: hea_ansatz(n, 1, t), th, dtype=dtype)
    obs = _terms(n, rng)
    e = b.energies(*obs)
    for y in range(3):
        assert C.functionals.expectation(b.states.state(y), *obs)[0] == e[y]
