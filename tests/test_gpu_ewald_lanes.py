"""GPU: lattice points that carry no term of an Ewald sum, beside others in the
same wave: the point at the shift itself, in the plane and out of it, and points
at infinity. Tolerance: 1e-10 of the largest coefficient of the same n (a few
hundred terms of a few roundings each, which may cancel to a fiftieth)."""
import ctypes
import math

import numpy as np
import pytest
import scipy.integrate
import scipy.special

import ewald_common as ec

pytestmark = pytest.mark.gpu
TOL = 1e-10
LAT_2D_IN_3D = 34
K0 = ec.wavenumber(2.0).real
BETA = (0.2 * 2 * np.pi / ec.A_LAT, 0.1 * 2 * np.pi / ec.A_LAT)


def close(a, b, LE):
    assert np.all(np.isfinite(a.view(float)))
    for n in range(LE + 1):
        p, q = a[n * n:(n + 1) ** 2], b[n * n:(n + 1) ** 2]
        assert np.all(np.abs(p - q) <= TOL * np.max(np.abs(q))), n


def short(L, LE, tr, R, err):
    """sigma^S of every triple, shifts in any direction, by the library's launcher."""
    import qpms_amd
    nsc, up = (LE + 1) ** 2, qpms_amd.DeviceBuffer.from_array
    leg0 = up(np.ones(55))   # P_n^m(0): for sums in the plane only
    dt, dR, out, er = up(tr), up(R), up(np.zeros((len(tr), nsc), complex)), up(np.zeros((len(tr), nsc)))
    L.qh_launch_sigma_short.argtypes = [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p,
                                        ctypes.c_double, ctypes.c_void_p, ctypes.c_int] + [ctypes.c_void_p] * 3
    L.qh_launch_sigma_short(LE, 0, len(tr), dt.ptr, len(R), dR.ptr, ec.ETA, leg0.ptr, -1,
                            out.ptr, er.ptr if err else None, None)
    L.qpms_hip_sync()
    return out.to_array(complex, (len(tr), nsc)), er.to_array(float, (len(tr), nsc))


def short_exact(LE, T, R):
    """The defining sum, I_n by quadrature, the point at the shift left out."""
    k = complex(T[3], T[4])
    out = np.zeros((LE + 1) ** 2, complex)
    for d in R - T[5:8]:
        r = np.linalg.norm(d)
        if r == 0:
            continue
        phi, ph = math.atan2(d[1], d[0]), np.exp(1j * (T[:3] @ d))
        for n in range(LE + 1):
            # t = eta u: eta^{2n+1} int_1^inf u^{2n} exp(-(r eta u)^2 + (k / 2 eta u)^2) du
            def f(u):
                return u ** (2 * n) * np.exp(-(r * ec.ETA * u) ** 2 + (k / (2 * ec.ETA * u)) ** 2)
            top = 1 + 30 / (r * ec.ETA)
            I = sum(c * scipy.integrate.quad(lambda u: getattr(f(u), w), 1, top, epsabs=0, epsrel=1e-12, limit=200)[0]
                    for c, w in ((1, "real"), (1j, "imag")) if w == "real" or k.imag)
            base = -1j * (2 * ec.ETA / k) ** (n + 1) * ec.ETA ** n / math.sqrt(math.pi) * r ** n * I * ph
            for m in range(-n, n + 1):
                s = base * scipy.special.lpmv(abs(m), n, d[2] / r) * np.exp(1j * m * phi)
                out[n * (n + 1) + m] += -s if m < 0 and m % 2 else s
    return out


@pytest.mark.parametrize("LE", [3, 7, 9])
@pytest.mark.parametrize("loss", [0.0, 0.2])
@pytest.mark.parametrize("err", [False, True])
def test_shift_out_of_plane_beside_zero(gpu, LE, loss, err):
    """One batch of a zero shift and shifts along and off the axis, the origin among the points."""
    L = ec.lib_ewald()
    R = np.column_stack([ec.R_points(2), np.zeros(len(ec.R_points(2)))])
    s = 0.3 * ec.A_LAT
    tr = np.array([[*BETA, 0, K0, loss * K0, *sh] for sh in ((0, 0, 0), (0, 0, s), (s, -s, 0.5 * s))])
    got, ge = short(L, LE, tr, R, err)
    for g, T in zip(got, tr):
        close(g, short_exact(LE, T, R), LE)
    assert np.all(np.isfinite(ge))


@pytest.mark.parametrize("k", [K0, K0 * (1 + 0.1j)])
def test_public_sum_with_the_origin(gpu, k):
    """ewald3_sigma_short for a lattice not marked as xy only."""
    import qpms_amd
    L, LE = ec.lib_ewald(), 7
    cart2, cart3 = qpms_amd.cart2_t, qpms_amd.cart3_t
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    res = []
    for origin in (True, False):
        g = L.PGen_xyWeb_new(cart2(*ec.B1), cart2(*ec.B2), 1e-13, cart2(0, 0), 0, origin, 12.5 * ec.H_R, False)
        out, err = np.empty((LE + 1) ** 2, complex), np.empty((LE + 1) ** 2)
        L.ewald3_sigma_short(out.ctypes.data, err.ctypes.data, e3c, ec.ETA, qpms_amd.c_cplx.of(k), LAT_2D_IN_3D,
                             ctypes.byref(g), False, cart3(*BETA, 0), cart3(0, 0, 0))
        assert np.all(np.isfinite(err))
        res.append(out)
    ref = ec.oracle_sigma_short(LE, k, BETA, (0, 0), ec.R_points(12, False))
    close(res[0], ref, LE)
    close(res[1], ref, LE)
    L.qpms_ewald3_constants_free(e3c)


@pytest.mark.parametrize("n", [1, 700])
def test_points_at_infinity(gpu, n):
    """They carry nothing: the sums of the lists with and without them are the same."""
    import qpms_amd
    L, LE = ec.lib_ewald(), 7
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    nsc, up = (LE + 1) ** 2, qpms_amd.DeviceBuffer.from_array
    tr = np.array([[*BETA, 0, K0 * (1 + 1e-3 * i), 0, 0.3 * ec.A_LAT, 0.1 * ec.A_LAT, 0] for i in range(n)])
    R, K = ec.R_points(3), ec.K_points(6 * 2 * np.pi / ec.A_LAT)
    far = np.array([[np.inf, 0.0], [0.0, -np.inf]])
    res = []
    for r, q in ((R, K), (np.vstack([far, R]), np.vstack([far, K]))):
        r = np.column_stack([r, np.zeros(len(r))])
        dt, dR, dK = up(tr), up(r), up(np.ascontiguousarray(q))
        ss, sl = up(np.zeros((n, nsc), complex)), up(np.zeros((n, nsc), complex))
        L.qpms_hip_ewald3_sigma_batch_dev(e3c, ec.ETA, ec.AREA, n, dt.ptr, len(r), dR.ptr, len(q), dK.ptr, ss.ptr,
                                          sl.ptr, None)
        L.qpms_hip_sync()
        res.append((ss.to_array(complex, (n, nsc)), sl.to_array(complex, (n, nsc))))
    for a, b in zip(res[1], res[0]):
        for i in (0, n - 1):
            close(a[i], b[i], LE)
    L.qpms_ewald3_constants_free(e3c)


@pytest.mark.parametrize("n", [1, 2, 29, 58, 1001, 344, 2 ** 20 + 1, 3 * 10 ** 8])
def test_phase_next_to_multiples_of_half_pi(gpu, n):
    """One K point: the sum's lowest coefficient is i e^{i K s} times a real number.
    Both parts of the phase to a few units in the last place of their own."""
    import qpms_amd
    L, LE = ec.lib_ewald(), 3
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    nsc, up = (LE + 1) ** 2, qpms_amd.DeviceBuffer.from_array
    x = n * (math.pi / 2)
    dt, dK, sl = up(np.array([[0, 0, 0, x / 10, 0, 1.0, 0, 0]])), up(np.array([[x, 0.0]])), up(np.zeros(nsc, complex))
    L.qpms_hip_ewald3_sigma_batch_dev(e3c, x / 4, 1.0, 1, dt.ptr, 0, dK.ptr, 1, dK.ptr, None, sl.ptr, None)
    L.qpms_hip_sync()
    v = sl.to_array(complex, (nsc,))[0] / 1j
    v /= np.copysign(abs(v), v.real * math.cos(x))
    assert abs(v.real / math.cos(x) - 1) < 2e-15 and abs(v.imag / math.sin(x) - 1) < 2e-15
    L.qpms_ewald3_constants_free(e3c)
