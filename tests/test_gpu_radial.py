"""The short-range space-charge solver over its radial grid sizes (its rows
are one per thread: below, at and above a wavefront, up to the largest grid,
and sizes that are no power of two) and modes, against the oracle."""
import numpy as np
import pytest

import cases
import g4mi
import harness as H

pytestmark = pytest.mark.gpu

COUNTS = [1024, 64, 256, 768]


@pytest.mark.parametrize("nz,nphi", [(1, 0), (2, 1)])
@pytest.mark.parametrize("ngr", [3, 4, 5, 63, 64, 65, 100, 129, 255, 256])
def test_radial_grids(ngr, nz, nphi):
    """FP64 form, separate, fused and split kernels: the on-axis field and the
    energies after two steps (the oracle's recurrence and the reduction are
    two orders of the same eliminations: 1e-12)."""
    st = H.steps(1, 2)[:2]
    sim = H.make_state(COUNTS, ngrid=41, sc=(nz, nphi, ngr, 0.0), seed_power=1e6)
    ctxs = []
    for fused in (0, 1, -1):
        ctx = H.to_gpu(sim)
        ctx.set_schedule("fp64_fused", fused)
        ctx.run(H.gsteps(st), cases.GAMMA0, record=())
        ctxs.append(ctx)
    sim.run(st, cases.GAMMA0, record=("power",))
    for ctx in ctxs:
        g = ctx.download_beam()["gamma"]
        assert np.max(np.abs(g - sim.gamma)) < 1e-12 * np.max(sim.gamma)
        assert H.rel_err(ctx.diag()["sscfield"], sim.sc_efield, 1e-12) < 1e-12
        ctx.close()


@pytest.mark.parametrize("ngr", [3, 64, 65, 129, 256])
def test_radial_grids_mixed(ngr):
    """Mixed form: FP32 positions pick the cells, so a particle may change
    its cell; one of 1024 moves the on-axis field by up to 1/1024 of a
    cell's charge, the bar the form's other space-charge test has (1e-3) for
    the largest slice and this share of the smaller ones."""
    st = H.steps(1, 2)[:1]
    sim = H.make_state([1024] * 3, ngrid=41, sc=(1, 0, ngr, 0.0), seed_power=1e6)
    ctx = H.to_gpu(sim, precision=g4mi.FP32)
    ctx.run(H.gsteps(st), cases.GAMMA0, record=())
    sim.run(st, cases.GAMMA0, record=("power",))
    e = H.rel_err(ctx.diag()["sscfield"], sim.sc_efield, 1e-12)
    print(f"  {ngr} radial cells: on-axis field {e:.2e}", flush=True)
    ctx.close()
    assert e < 1e-3
