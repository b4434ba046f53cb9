"""GPU: rounding errors of the triangular solves, and entries at the limits of the
range, for columns with a wave each (up to four) and with 16 lanes each."""
import ctypes

import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu


def solve(LU, B, prec=64):
    import qpms_amd
    L = qpms_amd.lib()
    L.qh_getrs_wait.argtypes = [ctypes.c_int] * 4 + [ctypes.c_void_p] * 3 + [ctypes.c_ulonglong, ctypes.c_void_p]
    dt = np.complex128 if prec == 64 else np.complex64
    n, nrhs = B.shape
    dA, dB, dp = [qpms_amd.DeviceBuffer.from_array(v)
                  for v in (LU.astype(dt), B.astype(dt), np.arange(n, dtype=np.int32))]
    L.qh_getrs_wait(prec, n, nrhs, 1, dA.ptr, dp.ptr, dB.ptr, 10 ** 7, None)
    return dB.to_array(dt, (n, nrhs))


def substitute(LU, B):
    """Column by column, in B's precision."""
    X = B.copy()
    with np.errstate(all="ignore"):
        for i in range(len(X)):
            X[i + 1:] -= LU[i + 1:, i:i + 1] * X[i]
        for i in range(len(X) - 1, -1, -1):
            X[i] /= LU[i, i]
            X[:i] -= LU[:i, i:i + 1] * X[i]
    return X


def system(n, nrhs, seed, kind):
    rng = np.random.default_rng(seed)
    A = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    if kind == "cluster":   # I - T W of weak scatterers
        A = np.eye(n) - A / (2.5 * np.sqrt(n)) * 10.0 ** rng.uniform(-3, 0, n)[:, None]
    if kind == "singular":   # condition 1e12
        A[:, n // 2] = A[:, :n // 2] @ rng.normal(size=n // 2) + 1e-12 * A[:, n // 2]
    return scipy.linalg.lu_factor(A)[0], rng.normal(size=(n, nrhs)) + 1j * rng.normal(size=(n, nrhs))


@pytest.mark.parametrize("kind", ["random", "cluster"])
@pytest.mark.parametrize("n, nrhs", [(64, 1), (64, 8), (200, 1), (200, 8), (512, 1), (512, 8)])
def test_error_of_substitution(gpu, n, nrhs, kind):
    """No larger than that of substitution column by column: the mean (of the
    logarithms) over 12 systems, each ratio spread by 1.4 or so, below 1.25."""
    ratio = []
    for seed in range(12):
        LU, B = system(n, nrhs, seed, kind)
        ref = substitute(LU.astype(np.clongdouble), B.astype(np.clongdouble))
        e = [float(np.linalg.norm(X - ref)) for X in (solve(LU, B), substitute(LU, B))]
        ratio.append(e[0] / e[1])
    assert np.exp(np.mean(np.log(ratio))) < 1.25


@pytest.mark.parametrize("nrhs", [1, 8])
@pytest.mark.parametrize("n", [63, 65, 300])
def test_nearly_singular(gpu, n, nrhs):
    """Backward stable row by row: |L U x - b| within n eps of |L| |U| |x| in either
    sweep, a few roundings each for the complex products."""
    LU, B = system(n, nrhs, n, "singular")
    X = solve(LU, B).astype(np.clongdouble)
    M = LU.astype(np.clongdouble)
    Lo, U = np.tril(M, -1) + np.eye(n), np.triu(M)
    res = np.abs(Lo @ (U @ X) - B)
    assert np.all(res <= 8 * n * 2.0 ** -53 * (np.abs(Lo) @ (np.abs(U) @ np.abs(X))))


@pytest.mark.parametrize("nrhs", [1, 8])
@pytest.mark.parametrize("prec, e", [(64, 1000), (64, 510), (32, 120), (32, 62)])
def test_rows_at_the_limits(gpu, prec, e, nrhs):
    """Rows of U times powers of two, as far as 2^-e: the solution is the same but for
    what the rows' order of magnitude changes nothing in, roundings."""
    n = 150
    rng = np.random.default_rng(e)
    LU, B = system(n, nrhs, 5, "cluster")
    scale = np.where(rng.uniform(size=n) < 0.3, 2.0 ** -e, np.where(rng.uniform(size=n) < 0.3, 2.0 ** (e // 2), 1.0))
    U, Lo = np.triu(LU) * scale[:, None], np.eye(n)
    x = solve(np.tril(Lo, -1) + U, B * scale[:, None], prec)
    ref = scipy.linalg.solve_triangular(np.triu(LU), B)
    eps = 2.0 ** -52 if prec == 64 else 2.0 ** -23
    assert np.max(np.abs(x - ref)) < 64 * np.sqrt(n) * eps * np.max(np.abs(ref))


@pytest.mark.parametrize("nrhs", [2, 8])
@pytest.mark.parametrize("k", [0, 20, 63, 70, 149])
def test_zero_pivot_and_nan(gpu, nrhs, k):
    """A zero on U's diagonal leaves the rows below alone; a NaN in one column leaves
    the other columns as they are without it."""
    LU, B = system(150, nrhs, 7, "cluster")
    x0 = solve(LU, B)
    C = B.copy()
    C[k, 1] = np.nan
    x1 = solve(LU, C)
    keep = np.arange(nrhs) != 1
    assert np.array_equal(x1[:, keep], x0[:, keep]) and not np.any(np.isfinite(x1[:, 1]))
    LU[k, k] = 0
    x2 = solve(LU, B)
    assert np.array_equal(x2[k + 1:], x0[k + 1:]) and not np.any(np.isfinite(x2[:k + 1]))
