"""GPU: the triangular solves (k_tri) at the edges of their 64-row blocks and
16-column slabs, with fewer workgroups than blocks, in batches, and left to one
workgroup; rows permuted by pivots alone."""
import ctypes

import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (15, 2, 1), (63, 16, 2), (64, 1, 3), (65, 17, 1), (127, 5, 2), (129, 33, 1), (300, 64, 1),
          (1000, 1, 2), (1000, 15, 1), (200, 3, 70), (4500, 1, 1), (4500, 20, 1)]


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("wait", [10 ** 7, 0])
@pytest.mark.parametrize("n, nrhs, batch", SHAPES)
def test_solve_edges(gpu, prec, wait, n, nrhs, batch):
    """Triangles of random entries 1 / (2 sqrt n) beside diagonals of modulus 1 to 2:
    each sweep's condition is below 10, rounding errors add like a random walk, so
    the error stays below 64 sqrt(n) eps of the largest entry."""
    import qpms_amd
    L = qpms_amd.lib()
    L.qh_getrs_wait.argtypes = [ctypes.c_int] * 4 + [ctypes.c_void_p] * 3 + [ctypes.c_ulonglong, ctypes.c_void_p]
    dt, eps = (np.complex128, 2.3e-16) if prec == 64 else (np.complex64, 1.2e-7)
    rng = np.random.default_rng(n + nrhs)

    def draw(*s):
        return rng.uniform(-1, 1, s) + 1j * rng.uniform(-1, 1, s)
    LU = draw(batch, n, n) / (2 * np.sqrt(n))
    LU[:, range(n), range(n)] = rng.uniform(1, 2, (batch, n)) * np.exp(2j * np.pi * rng.uniform(size=(batch, n)))
    LU, B = LU.astype(dt), draw(batch, n, nrhs).astype(dt)
    perm = np.stack([rng.permutation(n) for _ in range(batch)]).astype(np.int32)
    dA, dB, dp = [qpms_amd.DeviceBuffer.from_array(v) for v in (LU, B, perm)]
    L.qh_getrs_wait(prec, n, nrhs, batch, dA.ptr, dp.ptr, dB.ptr, wait, None)
    X = dB.to_array(dt, (batch, n, nrhs))
    for b in range(batch):
        M = LU[b].astype(complex)
        y = scipy.linalg.solve_triangular(M, B[b][perm[b]].astype(complex), lower=True, unit_diagonal=True)
        x = scipy.linalg.solve_triangular(M, y)
        assert np.max(np.abs(X[b] - x)) < 64 * np.sqrt(n) * eps * np.max(np.abs(x))


@pytest.mark.parametrize("n", [1, 2, 31, 33, 64, 65, 500])
def test_rows_by_pivots(gpu, n):
    import qpms_amd
    L = qpms_amd.lib()
    rng = np.random.default_rng(n)
    ipiv = np.array([rng.integers(i, n) + 1 for i in range(n)], np.int32)
    B = np.arange(2 * n).reshape(n, 2) + 1j
    want = B.copy()
    for i, p in enumerate(ipiv):
        want[[i, p - 1]] = want[[p - 1, i]]
    dA, dp, dB = [qpms_amd.DeviceBuffer.from_array(v) for v in (np.eye(n, dtype=complex), ipiv, B.astype(complex))]
    L.qpms_hip_zgetrs_dev(ctypes.c_size_t(n), ctypes.c_size_t(2), dA.ptr, dp.ptr, dB.ptr, None)
    assert np.array_equal(dB.to_array(np.complex128, (n, 2)), want)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n, nrhs", [(70, 1024), (70, 1025), (200, 3000), (3, 1100000)])
def test_more_columns_than_one_launch_takes(gpu, prec, n, nrhs):
    """Every column is the one of a solve of its own, to rounding (condition below 10);
    the words' memory does not grow with the columns."""
    import qpms_amd
    L = qpms_amd.lib()
    dt, eps = (np.complex128, 2.3e-16) if prec == 64 else (np.complex64, 1.2e-7)
    rng = np.random.default_rng(n)
    LU = (rng.uniform(-1, 1, (n, n)) + 1j * rng.uniform(-1, 1, (n, n))) / (2 * np.sqrt(n))
    LU[range(n), range(n)] = rng.uniform(1, 2, n)
    B = rng.normal(size=(n, nrhs)) + 1j * rng.normal(size=(n, nrhs))
    dA, dB, dp = [qpms_amd.DeviceBuffer.from_array(v)
                  for v in (LU.astype(dt), B.astype(dt), np.arange(n, dtype=np.int32))]
    L.qh_getrs_wait.argtypes = [ctypes.c_int] * 4 + [ctypes.c_void_p] * 3 + [ctypes.c_ulonglong, ctypes.c_void_p]
    L.qh_getrs_wait(prec, n, nrhs, 1, dA.ptr, dp.ptr, dB.ptr, 10 ** 7, None)
    X = dB.to_array(dt, (n, nrhs))
    x = scipy.linalg.solve_triangular(LU, scipy.linalg.solve_triangular(LU, B, lower=True, unit_diagonal=True))
    assert np.max(np.abs(X - x)) < 64 * np.sqrt(n) * eps * np.max(np.abs(x))
    L.qh_getrs_ws_bytes.restype = ctypes.c_size_t
    assert L.qh_getrs_ws_bytes(prec, n, nrhs, 1) == L.qh_getrs_ws_bytes(prec, n, min(nrhs, 1024), 1)
