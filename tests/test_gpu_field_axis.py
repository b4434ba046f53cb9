"""GPU: the scattered field on the particles' axes (k_scattered_e) against the oracle."""
import numpy as np
import pytest

import oracle_ffi as of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lMax", [1, 2, 3, 4])
@pytest.mark.parametrize("k, J", [(1.2e7, 3), (1.2e7, 4), (1.2e7 + 2e5j, 3), (1.2e7, 1)])
def test_axis_and_coinciding_points(gpu, lMax, k, J):
    """Points on and within rounding of the particles' z axes, at both sides, where
    the angular functions' limits count; the outgoing field at a particle is NaN.
    Odd numbers of points and particles. Tolerance: 1e-11 of the field there (the
    angular functions near the axis lose nothing in this library; the oracle's, which
    divide by sin(theta), up to 1e-16 / 1e-5)."""
    import qpms_amd
    rng = np.random.default_rng(lMax)
    pos = rng.uniform(-1e-6, 1e-6, (7, 3))
    cv = rng.normal(size=(7, 2 * lMax * (lMax + 2))) + 1j * rng.normal(size=(7, 2 * lMax * (lMax + 2)))
    off = np.array([(0, 0, 1), (0, 0, -1), (1e-5, 0, 1), (0, -1e-5, -1), (1e-5, 1e-5, 1), (1, 0, 0), (0, -1, 0)])
    pts = (pos[:, None] + 3e-7 * off[None]).reshape(-1, 3)
    got = qpms_amd.scattered_E(lMax, pos, k, cv, pts, J=J)
    ref = of.scattered_E(lMax, pos, k, cv.ravel(), pts, J=J)
    assert np.max(np.abs(got - ref)) < 1e-11 * np.max(np.abs(ref))
    if J >= 3:
        assert np.all(np.isnan(qpms_amd.scattered_E(lMax, pos, k, cv, pos[:1], J=J)))
