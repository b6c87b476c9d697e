"""The particle kernels' sines and cosines over the whole range of phases:
bunching of single particles at phases near multiples of pi/2, tiny, large
and beyond the range of the two-part reduction, against the C library's."""
import math

import numpy as np
import pytest

import g4mi
import harness as H

pytestmark = pytest.mark.gpu

@pytest.mark.parametrize("scale", [0.0, 1e-9, 1.0, 1e3, 1e7, 1e13, 3.6e13, 1e14, 1e19, 1e40, 1e150, 1e300, np.inf])
def test_bunching_of_single_particles(scale):
    """One particle in each of 512 slices: the record's cos and sin are those
    of its phase, within an ulp of an exact reduction and the roundings of
    the polar form, whatever the phase's size (the reduction changes at
    2^45 = 3.5e13); of a phase that is no number they are none."""
    rng = np.random.default_rng(5)
    n = 512
    th = rng.uniform(-1, 1, n) * scale if np.isfinite(scale) else np.full(n, np.nan)
    if scale == 1.0:
        th[:8] = np.arange(-4, 4) * (np.pi / 2)
    if scale == 3.6e13:
        th[:8] = [s * v for s in (-1, 1) for v in (np.nextafter(2.0 ** 45, 0), 2.0 ** 45,
                                                   np.nextafter(2.0 ** 45, 1e99), 2.0 ** 46)]
    if scale == 1e300:
        # the double nearest to a multiple of pi/2, and the largest
        th[:4] = [6381956970095103 * 2.0 ** 797, -6381956970095103 * 2.0 ** 797, 1.7976931348623157e308, -1.7e308]
    if not np.isfinite(scale):
        th[:4] = [np.inf, -np.inf, np.inf, -np.inf]
    sim = H.make_state([4] * n)
    sim.theta[:] = np.repeat(th, 4)
    ctx = H.to_gpu(sim)
    d = ctx.diag()
    ctx.close()
    if not np.isfinite(scale):
        assert np.all(np.isnan(d["bunching"]))
        return
    assert np.max(np.abs(d["bunching"] - 1)) < 8e-16
    z = np.exp(1j * d["bunchingphase"]) - np.array([complex(math.cos(t), math.sin(t)) for t in th])
    assert np.max(np.abs(z)) < 8e-16
