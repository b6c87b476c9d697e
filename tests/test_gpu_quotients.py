"""The FP64 particle kernels' quotients and square roots: in a drift without
a field every coordinate follows from products, quotients and roots alone, so
the three forms of the particle passes give the oracle's bits, also for
operands that have overflowed or vanished."""
import numpy as np
import pytest

import cases
import harness as H

pytestmark = pytest.mark.gpu
BEAM = ("gamma", "theta", "x", "y", "px", "py")
FORMS = {"fused": 1, "split": -1, "separate": 0}


KINDS = {"drift": lambda s: s.aw == 0 and s.qf == 0, "undulator": lambda s: s.aw > 0 and s.qf == 0,
         "quadrupole": lambda s: s.qf != 0}


def _step(sim, form, kind="drift"):
    st = H.steps(2, 3)
    one = [s for s in st if KINDS[kind](s)][:1]
    one[0].phaseshift = one[0].cx = one[0].cy = 0.0
    ctx = H.to_gpu(sim)
    ctx.set_schedule("fp64_fused", FORMS[form])
    assert ctx.schedule()["particle_passes"] == form
    ctx.run(H.gsteps(one), cases.GAMMA0, record=())
    sim.run(one, cases.GAMMA0, record=("power",))
    b = ctx.download_beam()
    ctx.close()
    return b


@pytest.mark.parametrize("form", FORMS)
def test_bits_of_a_drift(form):
    """Energies from rest to 1e70, momenta from 1e-250 to almost the whole
    energy: 400 000 quotients by gamma_z, gamma^2 and beta_par each, and as
    many roots, are the correctly rounded ones."""
    rng = np.random.default_rng(11)
    sim = H.make_state([4096] * 96, ngrid=31, timerun=False)
    n = len(sim.gamma)
    sim.gamma[:] = 1 + 10.0 ** rng.uniform(-6, 5, n)
    sim.gamma[::16] = 10.0 ** rng.uniform(5, 70, len(sim.gamma[::16]))
    u = np.sqrt(sim.gamma ** 2 - 1)
    for k, frac in (("px", 0.7), ("py", 0.7)):
        p = getattr(sim, k)
        p[:] = u * rng.uniform(-frac, frac, n)
        p[::2] = (rng.choice([-1, 1], n) * 10.0 ** np.minimum(rng.uniform(-250, 0, n), np.log10(u) - 1))[::2]
        getattr(sim, k[1])[:] = rng.normal(size=n) * 1e-4 * (rng.random(n) < 0.5)
    sim.theta[:] = rng.uniform(-1, 1, n)
    b = _step(sim, form)
    for k in BEAM:
        same = b[k] == getattr(sim, k)
        assert np.all(same), (k, int(np.sum(~same)), b[k][~same][:3], getattr(sim, k)[~same][:3])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("form", FORMS)
def test_operands_that_overflowed(form, kind):
    """Particles at rest or beyond, of infinite energy, momentum or position:
    each coordinate is the number, infinity or NaN that IEEE arithmetic gives
    (numbers to a few roundings, 1e-14, where sines enter), and the other
    particles of their slices are untouched."""
    inf, nan = np.inf, np.nan
    odd = [dict(gamma=inf), dict(gamma=1e200), dict(gamma=1e160, px=1e10), dict(gamma=1.25, px=0.75, py=0.0),
           dict(gamma=1.0, px=0.0, py=0.0), dict(gamma=0.5), dict(gamma=0.0), dict(px=inf), dict(px=1e300),
           dict(gamma=inf, px=1e300), dict(x=inf), dict(x=-inf, y=nan), dict(px=nan), dict(gamma=nan)]
    sim = H.make_state([512] * len(odd), ngrid=31, timerun=False)
    for i, o in enumerate(odd):
        for k, v in o.items():
            getattr(sim, k)[512 * i + 37] = v
    b = _step(sim, form, kind)
    for k in BEAM:
        ref = getattr(sim, k)
        same = (b[k] == ref) | (np.isnan(b[k]) & np.isnan(ref))
        num = np.isfinite(b[k]) & np.isfinite(ref)
        if kind != "drift":
            typ = np.median(np.abs(ref[num]))
            same[num] = np.abs(b[k][num] - ref[num]) <= 1e-14 * np.maximum(np.abs(ref[num]), typ)
        assert np.all(same), (k, [(odd[j // 512], b[k][j], ref[j]) for j in np.flatnonzero(~same)[:4]])
