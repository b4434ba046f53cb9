"""GPU: translation matrices built whole (several indices y per workgroup where
particles are many) against the same rows built one particle at a time (one y per
workgroup): the same arithmetic, so the same bits. Particle counts around the 64
sources of a wave and the numbers of workgroups at which the split changes."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lMax, npart", [(1, 1), (1, 171), (1, 700), (2, 64), (2, 65), (2, 256), (3, 34), (3, 69),
                                         (3, 150), (4, 21), (4, 43), (4, 64), (4, 100)])
def test_rows_of_whole_matrix(gpu, lMax, npart):
    import qpms_amd
    calc = qpms_amd.TransCalculator(lMax)
    L = qpms_amd.lib()
    g = np.random.default_rng(npart)
    pos = g.uniform(-1, 1, (npart, 3)) * 1e-6 * npart
    nb = 2 * lMax * (lMax + 2)
    W = calc.build_W(pos, 1.3e7).reshape(npart, nb, npart * nb)
    dpos, dW = qpms_amd.DeviceBuffer.from_array(pos), qpms_amd.DeviceBuffer(nb * npart * nb * 16)
    k = qpms_amd.c_cplx.of(1.3e7)
    for p in sorted({0, npart // 3, npart // 2, npart - 1}):
        L.qpms_hip_build_translation_matrix_rows_dev(calc.c, npart, dpos.ptr, k, qpms_amd.HANKEL_PLUS, p, 1, dW.ptr,
                                                    npart * nb, None)
        L.qpms_hip_sync()
        assert np.array_equal(dW.to_array(np.complex128, (nb, npart * nb)), W[p])


@pytest.mark.parametrize("lMax, npts", [(1, 1), (2, 1), (4, 1), (3, 65), (2, 8192), (2, 8200), (4, 3000)])
def test_batches_of_pairs(gpu, lMax, npts):
    """A batch's arrays against those of its points in batches of one."""
    import qpms_amd
    calc = qpms_amd.TransCalculator(lMax)
    g = np.random.default_rng(npts)
    kr, th, ph = g.uniform(1, 30, npts) + 0j, g.uniform(0, np.pi, npts), g.uniform(-3, 3, npts)
    A, B = calc.get_AB_arrays_batch(kr, th, ph)
    for i in sorted({0, npts // 2, npts - 1}):
        a, b = calc.get_AB_arrays_batch(kr[i:i + 1], th[i:i + 1], ph[i:i + 1])
        assert np.array_equal(a[0], A[i]) and np.array_equal(b[0], B[i])
