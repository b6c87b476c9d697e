"""The FP64 push over the whole range of phases its sines and cosines take:
bunching of single particles at phases near multiples of pi/2, tiny, large
and beyond the range of the two-part reduction, against numpy's."""
import numpy as np
import pytest

import g4mi
import harness as H

pytestmark = pytest.mark.gpu

@pytest.mark.parametrize("scale,tol", [(0.0, 4e-16), (1e-9, 4e-16), (1.0, 4e-16), (1e3, 4e-16), (1e7, 4e-16),
                                       (1e13, 4e-16), (1e14, 0.25), (1e300, None), (np.inf, None)])
def test_bunching_of_single_particles(scale, tol):
    """One particle in each of 64 slices: the record's cos and sin are those
    of its phase.  Below 2^45 rad within 0.93 ulp of an exact reduction and
    one rounding of the polar form; above, within twice the spacing of
    neighbouring phases (0.016 rad at 1e14, doubled for the modulus' own);
    beyond that finite and at most 1 in size, as any sine."""
    rng = np.random.default_rng(5)
    n = 64
    th = rng.uniform(-1, 1, n) * scale if np.isfinite(scale) else np.full(n, np.nan)
    if scale == 1.0:
        th[:8] = np.arange(-4, 4) * (np.pi / 2)
    sim = H.make_state([4] * n)
    sim.theta[:] = np.repeat(th, 4)
    ctx = H.to_gpu(sim)
    d = ctx.diag()
    ctx.close()
    if not np.isfinite(scale):
        assert np.all(np.isnan(d["bunching"]))
        return
    assert np.max(np.abs(d["bunching"] - 1)) < 8e-16
    if tol is not None:
        z = np.exp(1j * d["bunchingphase"]) - (np.cos(th) + 1j * np.sin(th))
        assert np.max(np.abs(z)) < 2 * tol
