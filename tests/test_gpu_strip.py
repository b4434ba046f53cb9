"""GPU: the partial-pivoting strips (k_strip) at the edges of their rows and
columns: orders around the 32-column strip, the 4-column chunk, the 64 rows of
a wave and the 256 (FP64) or 512 (FP32) rows of a workgroup, the strip left to
one workgroup, and entries that are no finite numbers."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def getrf_pp(A, prec, wait):
    import qpms_amd
    L = qpms_amd.lib()
    L.qh_getrf_pp.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                              ctypes.c_ulonglong, ctypes.c_void_p]
    dt = np.complex128 if prec == 64 else np.complex64
    n = len(A)
    dA = qpms_amd.DeviceBuffer.from_array(A.astype(dt))
    dp, di = qpms_amd.DeviceBuffer(4 * n), qpms_amd.DeviceBuffer(4)
    L.qh_getrf_pp(prec, n, dA.ptr, dp.ptr, di.ptr, wait, None)
    L.qpms_hip_sync()
    return dA.to_array(dt, (n, n)), dp.to_array(np.int32, (n,)), int(di.to_array(np.int32, (1,))[0])


def eliminate(A):
    """zgetf2: (LU, 1-based pivots); a column's pivot is its first row of largest
    |re| + |im|, rows that are no number last."""
    A = A.copy()
    n = len(A)
    piv = np.zeros(n, int)
    with np.errstate(all="ignore"):
        for j in range(n):
            mag = np.abs(A[j:, j].real) + np.abs(A[j:, j].imag)
            p = j + int(np.argmax(np.where(np.isnan(mag), -1.0, mag)))
            piv[j] = p + 1
            A[[j, p]] = A[[p, j]]
            mag = abs(A[j, j].real) + abs(A[j, j].imag)
            if mag > 0:
                A[j + 1:, j] = A[j + 1:, j] / A[j, j]
                A[j + 1:, j + 1:] -= np.multiply.outer(A[j + 1:, j], A[j, j + 1:])
    return A, piv


@pytest.mark.parametrize("wait", [10 ** 7, 0])
@pytest.mark.parametrize("prec, n", [(64, n) for n in (1, 3, 4, 5, 31, 32, 33, 36, 63, 65, 255, 256, 257, 289, 600)]
                         + [(32, n) for n in (1, 6, 33, 64, 65, 511, 512, 513, 545, 1100)])
def test_strip_edges(gpu, prec, n, wait):
    rng = np.random.default_rng(n)
    A = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    A = A.astype(np.complex64).astype(complex) if prec == 32 else A
    LU, piv, info = getrf_pp(A, prec, wait)
    assert info == 0
    if prec == 64:
        ref, rp = eliminate(A)
        assert np.array_equal(piv, rp)
        assert np.max(np.abs(LU - ref)) < 1e-13 * n * np.max(np.abs(ref))
    # P A = L U to rounding (n products of each entry), multipliers bounded by the pivot rule
    LU = LU.astype(complex)
    Lo, U, PA = np.tril(LU, -1) + np.eye(n), np.triu(LU), A.copy()
    for i, p in enumerate(piv - 1):
        PA[[i, p]] = PA[[p, i]]
    eps = 2.0 ** -52 if prec == 64 else 2.0 ** -23
    assert np.max(np.abs(Lo @ U - PA)) < 8 * eps * n * np.max(np.abs(U))
    assert np.max(np.abs(Lo)) < np.sqrt(2) * (1 + 64 * eps)


def test_strip_zero_pivot(gpu):
    A = np.random.default_rng(3).normal(size=(40, 40)) + 0j
    A[:, 7] = A[:, 2] = 0.0
    LU, piv, info = getrf_pp(A, 64, 10 ** 7)
    assert info == 3 and piv[2] == 3
    assert np.all(LU[3:32, 2] == 0) and np.all(np.isfinite(LU))


@pytest.mark.parametrize("where", [[(5, 20, np.inf)], [(17, 9, np.nan)], [(0, 31, np.nan), (30, 1, np.inf)],
                                   [(12, 12, -np.inf), (13, 29, np.nan)]])
def test_strip_non_finite(gpu, where):
    """What an infinity or NaN reaches, and what it leaves alone, as column by column."""
    A = np.random.default_rng(11).normal(size=(32, 32)) + 1j * np.random.default_rng(12).normal(size=(32, 32))
    for r, c, v in where:
        A[r, c] = v
    LU, piv, info = getrf_pp(A, 64, 10 ** 7)
    ref, rp = eliminate(A)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(LU), fin)
    assert fin.sum() > 200
    assert np.max(np.abs(LU[fin] - ref[fin])) < 1e-11 * np.max(np.abs(ref[fin]))
    ok = int(np.argmin(np.append(fin.all(axis=0), False)))   # columns before the first that is touched
    assert np.array_equal(piv[:ok], rp[:ok])


@pytest.mark.parametrize("prec, n", [(64, 32), (64, 64), (64, 512), (32, 64), (32, 1024)])
def test_strip_ties(gpu, prec, n):
    """A Hadamard matrix: every pivot search is a tie of many rows, and every
    value a power of two, so that the first row has to win each time."""
    H = np.ones((1, 1))
    while len(H) < n:
        H = np.block([[H, H], [H, -H]])
    LU, piv, info = getrf_pp(H + 0j, prec, 10 ** 7)
    ref, rp = eliminate(H + 0j)
    assert info == 0 and np.array_equal(piv, rp) and np.array_equal(LU, ref)


def test_blocks_by_tournament(gpu):
    """Blocks of more rows than the strips' workgroups find CUs for beside the
    trailing update (FP64: 8192) go by tournament, the others by k_strip."""
    import qpms_amd
    from test_gpu_lu import check_plu
    L = qpms_amd.lib()
    n = 8800
    rng = np.random.default_rng(5)
    A = np.empty((n, n), np.complex128)
    A.real = rng.random((n, n), np.float32) - 0.5
    A.imag = rng.random((n, n), np.float32) - 0.5
    dA = qpms_amd.DeviceBuffer.from_array(A)
    dp, dq, di = qpms_amd.DeviceBuffer(4 * n), qpms_amd.DeviceBuffer(4 * n), qpms_amd.DeviceBuffer.from_array(
        np.zeros(1, np.int32))
    L.qh_getrf_batched_f64.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_long, ctypes.c_void_p,
                                       ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    L.qh_getrf_batched_f64(n, 1, dA.ptr, n * n, dp.ptr, dq.ptr, di.ptr, None)
    L.qpms_hip_sync()
    assert int(di.to_array(np.int32, (1,))[0]) == 0
    # rows of a random matrix: |L| <= 2 or so per level of the tournament, errors of n products
    check_plu(A, dA.to_array(np.complex128, (n, n)), dp.to_array(np.int32, (n,)), 1e-13)


@pytest.mark.parametrize("n", [30, 100, 260])
@pytest.mark.parametrize("wait", [10 ** 7, 0])
def test_error_of_elimination(gpu, n, wait):
    """Errors of the factors of I - T W of weak scatterers no larger than those of
    elimination column by column: the mean (of the logarithms) over 6 systems, each
    ratio spread by 1.2 or so, below 1.15."""
    ratio = []
    for seed in range(6):
        rng = np.random.default_rng(seed)
        A = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        A = np.eye(n) - A / (2.5 * np.sqrt(n)) * 10.0 ** rng.uniform(-3, 0, n)[:, None]
        LU, piv, _ = getrf_pp(A, 64, wait)
        plain, rp = eliminate(A)
        ref, xp = eliminate(A.astype(np.clongdouble))
        assert np.array_equal(piv, xp) and np.array_equal(rp, xp)
        ratio.append(float(np.linalg.norm(LU - ref) / np.linalg.norm(plain - ref)))
    assert np.exp(np.mean(np.log(ratio))) < 1.15
