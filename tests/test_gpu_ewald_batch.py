"""GPU: the batched Ewald sums against the same triples one at a time: workgroups
of several waves per triple, of one, kernels by kind of wavenumber, both sums in
one launch, and many shifts of one (beta, k). Point counts around the 64 lanes and
the waves of a workgroup. Tolerance: 1e-10 of the triple's largest coefficient of
the same n (2435 terms of a few roundings each, which may cancel to a fiftieth)."""
import ctypes

import numpy as np
import pytest

import ewald_common as ec

pytestmark = pytest.mark.gpu
TOL = 1e-10


def triples(n, rng):
    k0, s = ec.wavenumber(2.0), ec.A_LAT / np.sqrt(3)
    t = np.zeros((n, 8))
    t[:, :2] = rng.uniform(-0.4, 0.4, (n, 2)) * 2 * np.pi / ec.A_LAT
    t[:, 3] = k0.real * rng.uniform(0.8, 1.2, n)
    t[:, 4] = np.where(rng.uniform(size=n) < 0.4, 1e-3 * k0.real, 0.0)
    t[:, 5] = rng.choice([0.0, s, -s], n)
    return t


def points(nR, nK):
    L = ec.lib_ewald()
    R, K = ec.R_points(), ec.K_points()
    R = R[np.argsort(np.hypot(*R.T), kind="stable")][:nR]
    K = K[np.argsort(np.hypot(*K.T), kind="stable")][:nK]
    return L, np.column_stack([R, np.zeros(len(R))]), K


def batch(L, e3c, LE, t, R, K, what="both"):
    import qpms_amd
    nsc = (LE + 1) ** 2
    up = qpms_amd.DeviceBuffer.from_array
    dt, dR, dK = up(t), up(R if len(R) else np.zeros((1, 3))), up(K if len(K) else np.zeros((1, 2)))
    ds, dl = up(np.full((len(t), nsc), np.nan + 0j)), up(np.full((len(t), nsc), np.nan + 0j))
    L.qpms_hip_ewald3_sigma_batch_dev(e3c, ec.ETA, ec.AREA, len(t), dt.ptr, len(R), dR.ptr, len(K), dK.ptr,
                                      ds.ptr if what != "long" else None, dl.ptr if what != "short" else None, None)
    L.qpms_hip_sync()
    return ds.to_array(complex, (len(t), nsc)), dl.to_array(complex, (len(t), nsc))


def close(a, b, LE):
    for n in range(LE + 1):
        p, q = a[:, n * n:(n + 1) ** 2], b[:, n * n:(n + 1) ** 2]
        assert np.all(np.abs(p - q) <= TOL * np.max(np.abs(q), axis=1, keepdims=True)), n


@pytest.mark.parametrize("LE", [3, 5, 7, 9])
@pytest.mark.parametrize("n, nR, nK", [(1, 433, 2435), (5, 0, 0), (5, 1, 1), (130, 63, 65), (300, 64, 513), (700, 433, 2435)])
def test_batch_against_single(gpu, LE, n, nR, nK):
    L, R, K = points(nR, nK)
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    t = triples(n, np.random.default_rng(n))
    ss, sl = batch(L, e3c, LE, t, R, K)
    some = sorted({0, 1 % n, n // 2, n - 1} | set(range(min(n, 8))))
    rs = np.vstack([batch(L, e3c, LE, t[i:i + 1], R, K, "short")[0] for i in some])
    rl = np.vstack([batch(L, e3c, LE, t[i:i + 1], R, K, "long")[1] for i in some])
    close(ss[some], rs, LE)
    close(sl[some], rl, LE)
    L.qpms_ewald3_constants_free(e3c)


@pytest.mark.parametrize("LE", [3, 5, 7, 9])
def test_one_sum_against_both(gpu, LE):
    """Enough triples for one wave each in launches of one sum; of both, and few."""
    L, R, K = points(70, 130)
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    t = triples(1100, np.random.default_rng(LE))
    ss, sl = batch(L, e3c, LE, t, R, K)
    close(batch(L, e3c, LE, t, R, K, "short")[0], ss, LE)
    close(batch(L, e3c, LE, t, R, K, "long")[1], sl, LE)
    few = t[:200]
    close(batch(L, e3c, LE, few, R, K, "short")[0], ss[:200], LE)
    close(batch(L, e3c, LE, few, R, K, "long")[1], sl[:200], LE)
    L.qpms_ewald3_constants_free(e3c)


@pytest.mark.parametrize("LE", [3, 5, 7, 9])
@pytest.mark.parametrize("n, nK", [(1, 2435), (63, 15), (65, 17), (300, 0), (300, 161)])
def test_shifts_against_single(gpu, LE, n, nK):
    import qpms_amd
    L, R, K = points(0, nK)
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    rng = np.random.default_rng(n)
    t = triples(n, rng)
    t[:, :5] = t[0, :5]
    t[:, 5:7] = rng.uniform(-2, 2, (n, 2)) * ec.A_LAT
    L.qh_ewald3_long_shifts_scratch.restype = ctypes.c_size_t
    L.qh_ewald3_long_shifts_scratch.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    L.qh_ewald3_sigma_long_shifts_dev.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_double, ctypes.c_size_t,
                                                  ctypes.c_void_p, ctypes.c_size_t] + [ctypes.c_void_p] * 4
    up, nsc = qpms_amd.DeviceBuffer.from_array, (LE + 1) ** 2
    dt, dK = up(t), up(K if len(K) else np.zeros((1, 2)))
    F = qpms_amd.DeviceBuffer(max(16, L.qh_ewald3_long_shifts_scratch(e3c, len(K))))
    out = up(np.full((n, nsc), np.nan + 0j))
    L.qh_ewald3_sigma_long_shifts_dev(e3c, ec.ETA, ec.AREA, n, dt.ptr, len(K), dK.ptr, F.ptr, out.ptr, None)
    L.qpms_hip_sync()
    got = out.to_array(complex, (n, nsc))
    some = sorted({0, n // 2, n - 1})
    close(got[some], np.vstack([batch(L, e3c, LE, t[i:i + 1], R, K, "long")[1] for i in some]), LE)
    L.qpms_ewald3_constants_free(e3c)


def test_more_triples_than_one_dispatch_takes(gpu):
    """2^25 + 3 triples in one call: the first, the last and those around 2^24."""
    import qpms_amd
    L, R, K = points(1, 1)
    e3c = L.qpms_ewald3_constants_init(3, -1)
    few, n, nsc = triples(1003, np.random.default_rng(1)), (1 << 25) + 3, 16
    up = qpms_amd.DeviceBuffer.from_array
    dt, dR, dK = up(np.resize(few, (n, 8))), up(R), up(K)
    ds, dl = qpms_amd.DeviceBuffer(16 * nsc * n), qpms_amd.DeviceBuffer(16 * nsc * n)
    L.qpms_hip_ewald3_sigma_batch_dev(e3c, ec.ETA, ec.AREA, n, dt.ptr, 1, dR.ptr, 1, dK.ptr, ds.ptr, dl.ptr, None)
    L.qpms_hip_sync()
    ss, sl = batch(L, e3c, 3, few, R, K)
    got = np.empty((2, nsc), complex)
    for t in (0, (1 << 24) - 2, 1 << 24, (1 << 25) - 1, n - 2):
        for d, ref in ((ds, ss), (dl, sl)):
            L.qpms_hip_memcpy_d2h(got.ctypes.data, d.ptr + 16 * nsc * t, got.nbytes)
            close(got, ref[[t % 1003, (t + 1) % 1003]], 3)
    L.qpms_ewald3_constants_free(e3c)
