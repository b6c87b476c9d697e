"""The tables kept per step size (ADI factors and bands, spectral kernels)
against the oracle: a line with more distinct step sizes than a context
keeps, walked twice so that every table is dropped and built again."""
import ctypes as C

import numpy as np
import pytest

import g4mi
import harness as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["adi", "fft"])
@pytest.mark.parametrize("ngrid", [31, 40])
def test_more_step_sizes_than_kept(solver, ngrid):
    sim = H.make_state([256] * 3, ngrid=ngrid, seed_power=1e4, timerun=False)
    if solver == "fft":
        sim.s.fft_solver = 1
    ctx = H.to_gpu(sim)
    ctx.set_field_solver(fft=solver == "fft")
    st = H.steps(1, 2)
    one = H.gsteps(st)[0]
    for k in [i % 36 for i in range(74)]:
        delz = 0.01 * (1 + 0.5 * k)
        ctx.field_track(one, delz)
        H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
    f, _ = ctx.download_field()
    err = np.max(np.abs(f - sim.field)) / np.max(np.abs(sim.field))
    print(f"  {solver} {ngrid}^2, 36 step sizes twice: {err:.2e}", flush=True)
    assert err < 1e-11  # 74 steps of the single step's 1e-13 bar
    ctx.close()
