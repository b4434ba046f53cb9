"""GPU: the Ewald sums of every order against the oracle, which sums in extended
precision, for real wavenumbers and complex ones with Im k up to Re k."""
import math

import numpy as np
import pytest

import ewald_common as ec
from test_gpu_ewald_batch import batch, close

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.mark.parametrize("LE", [3, 5, 7, 9])
@pytest.mark.parametrize("loss", [0.0, 1e-3, 0.1, 0.3])
@pytest.mark.parametrize("eV", [0.7, 2.0, 4.0])
def test_lattice_sums(gpu, LE, loss, eV):
    """19 R points, 313 K points from below the light cone to underflow, at shifts
    zero and not; k up to 2.4 times 2 eta (the terms grow as e^{(k / 2 eta)^2}, and at
    3.5 what is left of them has lost eight digits in any double arithmetic)."""
    L = ec.lib_ewald()
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    k = ec.wavenumber(eV) * (1 + 1j * loss)
    beta, s = (0.21 * 2 * np.pi / ec.A_LAT, 0.13 * 2 * np.pi / ec.A_LAT), (0.3 * ec.A_LAT, -0.2 * ec.A_LAT)
    R, K = ec.R_points(2), ec.K_points(12.5 * 2 * np.pi / ec.A_LAT)
    t = np.array([[*beta, 0, k.real, k.imag, *sh, 0] for sh in ((0, 0), s)])
    ss, sl = batch(L, e3c, LE, t, np.column_stack([R, np.zeros(len(R))]), K)
    R0 = R[np.hypot(*R.T) > 0]
    close(ss, np.array([ec.oracle_sigma_short(LE, k, beta, (0, 0), R0), ec.oracle_sigma_short(LE, k, beta, s, R)]), LE)
    close(sl, np.array([ec.oracle_sigma_long(LE, k, beta, sh, K) for sh in ((0, 0), s)]), LE)
    L.qpms_ewald3_constants_free(e3c)


def gamma_terms(LE, k, rb, eta):
    """Of one K point: per (n, |m|) the sum of the moduli of the terms in j; |z|."""
    from scipy.special import gamma
    import ctypes

    import oracle_ffi as of
    o = of.oracle()
    o.or_gamma_inc.restype = of.c_cplx
    o.or_gamma_inc.argtypes = [ctypes.c_double, of.c_cplx, ctypes.c_int]
    t = rb / k
    g = np.sqrt(t - 1) * np.sqrt(t + 1)
    z = (g * k / (2 * eta)) ** 2
    G = [abs(complex(v.re, v.im)) for v in (o.or_gamma_inc(0.5 - j, of.c_cplx.of(z), 0) for j in range(LE // 2 + 1))]
    out = np.zeros((LE + 1) ** 2)
    for n in range(LE + 1):
        for m in range(-n, n + 1, 2):
            a, b = (n - abs(m)) // 2, (n + abs(m)) // 2
            p0 = math.prod(range(n + abs(m) - 1, 1, -2)) / math.prod(range(n - abs(m), 1, -2))
            out[n * (n + 1) + m] = p0 * sum(
                gamma(a + 1) * gamma(b + 1) / (gamma(j + 1) * gamma(a - j + 1) * gamma(b - j + 1))
                * abs(t) ** (n - 2 * j) * abs(g) ** (2 * j - 1) * G[j] for j in range(a + 1))
    return out * 2 * math.sqrt(math.pi) / (abs(k) ** 2 * ec.AREA), abs(z)


@pytest.mark.parametrize("LE", [3, 5, 7, 9])
@pytest.mark.parametrize("loss", [0.01, 0.3, 1.0])
def test_incomplete_gamma_functions(gpu, LE, loss):
    """One K point, |z| from 0.3 to 44 to either side of Re z = 0.5: every coefficient
    within 100 roundings of its terms, and 4 of z, whose error e^{-z} takes on."""
    L = ec.lib_ewald()
    e3c = L.qpms_ewald3_constants_init(LE, -1)
    eta, tr = ec.ETA, []
    for kr in (0.5, 2.0, 4.0, 8.0):
        k = kr * eta * (1 + 1j * loss)
        for rez in (0.3, 0.51, 1.0, 3.0, 10.0, 30.0):
            rb2 = 4 * rez * eta ** 2 + (k * k).real
            if rb2 > 0:
                tr.append([math.sqrt(rb2) * math.cos(0.7), math.sqrt(rb2) * math.sin(0.7), 0, k.real, k.imag, 0, 0, 0])
    tr, K = np.array(tr), np.zeros((1, 2))
    _, got = batch(L, e3c, LE, tr, np.zeros((0, 3)), K)
    for t, g in zip(tr, got):
        k = complex(t[3], t[4])
        ref = ec.oracle_sigma_long(LE, k, t[:2], (0, 0), K)
        terms, z = gamma_terms(LE, k, math.hypot(*t[:2]), eta)
        assert np.all(np.abs(g - ref) <= (100 + 4 * z) * EPS * terms)
    L.qpms_ewald3_constants_free(e3c)
