"""Exact sampling by tiles of 4096 elements: numpy's sequential cumsum bit for
bit, on inputs that cross binades, hold ties, zeros and subnormals at the
edges of tiles, for arrays and states."""
import numpy as np
import pytest

from helpers import device_state

pytestmark = pytest.mark.gpu


def _amplitudes(kind, n, rng):
    """Real amplitudes whose squares have the named structure (not normalised:
    choice divides by the last entry of the cumsum)."""
    N = 1 << n
    a = np.zeros(N)
    if kind == "random":
        a[:] = rng.standard_normal(N) * 2.0 ** (-n / 2)
    elif kind == "uniform":
        a[:] = 2.0 ** -(n // 2)
    elif kind == "ties":
        # |a|^2 = 2^-54 after a first entry near 1: p / ulp is 1/2, 1, 2, ...
        a[:] = 2.0 ** -27.0 * rng.choice([0.0, 0.5, 1.0, 2.0, 3.0], N)
        a[0] = 2.0 ** -0.5 + 2.0 ** -30
        a[N // 2] = 1.0
    elif kind == "zeros":  # GHZ-like: long runs of zeros, first entry past a tile's edge
        a[min(4096, N - 1)] = a[N - 1] = 2.0 ** -0.5
    elif kind == "tiny":  # subnormal sums that grow over hundreds of binades
        a[:] = 2.0 ** np.linspace(-537, -1, N)
    elif kind == "steps":  # c lands on powers of two at tile edges
        a[::4096] = 0.5
        a[1:8] = 2.0 ** -26
    return a


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("kind", ["random", "uniform", "ties", "zeros", "tiny", "steps"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 11, 12, 13, 16])
def test_exact_samples_by_tiles(C, n, kind, dtype):
    if kind == "tiny" and dtype == "complex64":
        pytest.skip("below complex64's range")
    rng = np.random.default_rng(17 * n)
    a = _amplitudes(kind, n, rng)
    sv = device_state(C, n, dtype, a.astype(dtype))
    u = np.concatenate([rng.random(3000), [0.0, 0.5, 0.25, 1 - 2.0 ** -53]])
    for normalize in (False, True):
        p = C.functionals.probabilities(sv, normalize=normalize)
        cdf = np.cumsum(p)
        want = np.searchsorted(cdf / cdf[-1], u, side="right")
        got = C.functionals.sample(sv, u, exact=True, normalize=normalize)
        assert np.array_equal(got, want), normalize


def test_more_tiles_than_one_scan(C):
    """2^23 elements: 2048 tiles, two scans of the chain, random and with a
    flat stretch at a power of two."""
    n = 23
    rng = np.random.default_rng(2)
    u = rng.random(20000)
    a = (rng.standard_normal(1 << n) * 2.0 ** (-n / 2)).astype(np.complex64)
    b = np.full(1 << n, 2.0 ** -40, np.complex64)
    b[0] = b[1 << 22] = 2.0 ** -0.5
    for v in (a, b):
        sv = device_state(C, n, "complex64", v)
        p = C.functionals.probabilities(sv, normalize=True)
        cdf = np.cumsum(p)
        want = np.searchsorted(cdf / cdf[-1], u, side="right")
        assert np.array_equal(C.functionals.sample(sv, u, exact=True, normalize=True), want)


def test_largest_state(C):
    """34 qubits complex64 (128 GiB): 2^22 tiles, whose threads one launch
    dimension does not hold.  H on the first, a middle and the last qubit gives
    eight equal entries."""
    n, item = 34, 8
    if C.core.cuda.mem_info()[0] < (item << n) + (1 << (n - 1)) + (4 << 30):
        pytest.skip("needs 140 GiB of free device memory")
    g = C.operation.gate_operations
    sv = device_state(C, n, "complex64")
    where = np.zeros(1, np.int64)
    for q in (0, 16, n - 1):
        C.functionals.apply(sv, g.Hadamard([q]), n, [q])
        where = np.concatenate([where, where | 1 << (n - 1 - q)])
    u = np.random.default_rng(5).random(500)
    # the entries differ in the last bits only: no uniform is that close to k / 8
    assert np.abs(8 * u - np.round(8 * u)).min() > 1e-5
    got = C.functionals.sample(sv, u, exact=True, normalize=True)
    assert np.array_equal(got, np.sort(where)[(8 * u).astype(int)])


def _library(C):
    import ctypes
    import os

    L = ctypes.CDLL(os.path.join(os.path.dirname(C.__file__), "libsnuqs_hip.so"))
    P, Q = ctypes.c_void_p, ctypes.c_uint64
    L.sq_sample.argtypes = [P, Q, P, Q, ctypes.c_int, P, P]
    L.sq_memcpy_h2d.argtypes = [P, P, ctypes.c_size_t, P]
    return L


# finite entries whose sum passes the largest double: at the last entry numpy's
# cdf ends in inf and every index is the last; before it the call is refused
@pytest.mark.parametrize("n,at", [(1, (0, 1)), (2, (0, 1)), (2, (1, 3)), (13, (10, 20)),
                                  (13, (10, 8000)), (23, (1 << 22, (1 << 22) + 5)),
                                  (23, (7, (1 << 23) - 1))])
def test_sums_past_the_range_of_doubles(C, n, at):
    L = _library(C)
    p = np.zeros(1 << n)
    p[list(at)] = 1.2e308
    buf = C.result_types.StateVector(C.DeviceType.CUDA, n, dtype="complex64")  # 8 bytes an entry
    u = np.array([0.0, 0.3, 0.9])
    out = np.full(3, -1, np.int64)
    assert L.sq_memcpy_h2d(buf.data_ptr, p.ctypes.data, p.nbytes, None) == 0
    rc = L.sq_sample(buf.data_ptr, 1 << n, u.ctypes.data, 3, 1, out.ctypes.data, None)
    if at[1] == (1 << n) - 1:
        assert rc == 0 and (out == (1 << n) - 1).all()
    else:
        assert rc == 1  # SQ_ERR_INVALID
    # the same from a state
    a = np.zeros(1 << n, np.complex128)
    a[list(at)] = 1.1e154  # squares to 1.21e308
    sv = device_state(C, n, "complex128", a)
    if at[1] == (1 << n) - 1:
        assert (C.functionals.sample(sv, u, exact=True) == (1 << n) - 1).all()
    else:
        with pytest.raises(ValueError):
            C.functionals.sample(sv, u, exact=True)


def test_negative_entries_through_the_c_abi(C):
    """An array with a negative entry still takes the older route (numpy
    refuses it; here it gives the cumsum's answer as before)."""
    L = _library(C)
    n = 13
    p = np.random.default_rng(1).random(1 << n) / (1 << n)
    p[5000] = -p[5000]
    buf = C.result_types.StateVector(C.DeviceType.CUDA, n, dtype="complex64")  # 8 bytes an entry
    u = np.random.default_rng(2).random(500)
    out = np.empty(500, np.int64)
    assert L.sq_memcpy_h2d(buf.data_ptr, p.ctypes.data, p.nbytes, None) == 0
    assert L.sq_sample(buf.data_ptr, 1 << n, u.ctypes.data, 500, 0, out.ctypes.data, None) == 0
    fast = out.copy()
    assert L.sq_sample(buf.data_ptr, 1 << n, u.ctypes.data, 500, 1, out.ctypes.data, None) == 0
    assert np.abs(out - fast).max() <= 1


def test_probabilities_are_given_back(C):
    """Fast sampling from a state keeps the cdf (8 bytes an element) and some
    scratch in the workspace, and not the probabilities."""
    n = 28
    sv = device_state(C, n, "complex64")
    u = np.random.default_rng(3).random(100)
    C.functionals.sample(sv, u, exact=True)

    def free():
        # (the runtime returns memory with the next allocation and release)
        other = C.result_types.StateVector(C.DeviceType.CUDA, n, dtype="complex64")
        del other
        return C.core.cuda.mem_info()[0]

    before = free()
    assert (C.functionals.sample(sv, u, exact=False) == 0).all()
    assert before - free() < 12 << n
