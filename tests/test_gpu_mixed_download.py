"""The mixed form's downloads, widened on the device piece by piece: every
value is the FP32 one exactly, over pieces that end inside slices and fields,
with empty slices and negative zeros."""
import numpy as np
import pytest

import g4mi
import harness as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,ngrid", [([0, 131068, 8, 0, 40000, 0], 31), ([140000, 4], 255), ([16], 15),
                                          ([1020, 2044, 512], 255)])
def test_downloads_are_the_fp32_values(counts, ngrid):
    sim = H.make_state(counts, ngrid=ngrid)
    rng = np.random.default_rng(len(counts))
    sim.theta += np.repeat(rng.integers(-40, 40, len(counts)), counts) * 7.0
    sim.x[::3] = -0.0
    sim.field[:] = rng.normal(size=sim.field.shape) * 1e9
    sim.field[:, ::5, 1] = -0.0
    ctx = H.to_gpu(sim, precision=g4mi.FP32)
    b = ctx.download_beam()
    f, _ = ctx.download_field()
    for k in ("x", "y", "px", "py"):
        want = getattr(sim, k).astype(np.float32).astype(np.float64)
        assert np.array_equal(b[k], want) and np.array_equal(np.signbit(b[k]), np.signbit(want)), k
    gref = np.float64(np.float32(sum(sim.gamma.tolist()) / len(sim.gamma)))
    assert np.array_equal(b["gamma"], gref + (sim.gamma - gref).astype(np.float32).astype(np.float64))
    for a, e in zip(sim.off[:-1], sim.off[1:]):
        if e > a:
            base = 2 * np.pi * np.floor(sum(sim.theta[a:e].tolist()) / (e - a) / (2 * np.pi))
            want = base + (sim.theta[a:e] - base).astype(np.float32).astype(np.float64)
            assert np.array_equal(b["theta"][a:e], want)
    want = sim.field.astype(np.float32).astype(np.float64)
    assert np.array_equal(f, want) and np.array_equal(np.signbit(f), np.signbit(want))
    ctx.close()
