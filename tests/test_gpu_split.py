"""The small-window step (particle passes over blocks of the particles, the
split deposit) against the oracle and against the fused kernels: sizes at the
edges of its blocks of 256 and chunks of 512 particles, empty slices, footprints
within and beyond the deposit's LDS tile, particles outside the grid, with and
without space charge, harmonic fields, a chicane, sorted and dropped
particles."""
import numpy as np
import pytest

import cases
import harness as H

pytestmark = pytest.mark.gpu
BEAM = ("gamma", "theta", "x", "y", "px", "py")


def _check(sim, ctx, st, tol=1e-12):
    g = ctx.run(H.gsteps(st), cases.GAMMA0, record=("power", "bunching", "energy", "xsize", "nf_intensity"))
    r = sim.run(st, cases.GAMMA0, record=("power", "bunching", "energy", "xsize", "nf_intensity"))
    for k in g:  # against the largest value: an unmodulated beam's bunching is a sum that cancels
        assert np.max(np.abs(g[k] - r[k])) <= 1e-10 * np.max(np.abs(r[k])), k
    b = ctx.download_beam()
    for k in BEAM:
        ref = getattr(sim, k)
        assert np.max(np.abs(b[k] - ref)) <= tol * np.max(np.abs(ref)), k
    f, first = ctx.download_field()
    assert first == sim.s.first
    assert np.max(np.abs(f - sim.field)) <= tol * np.max(np.abs(sim.field))


@pytest.mark.parametrize("sc", [(0, 0, 100, 0.0), (1, 0, 100, 0.0)])
@pytest.mark.parametrize("counts", [[4], [252, 0, 256, 260], [508, 512, 516, 8196], [0, 0, 1028, 0]])
def test_block_edges(counts, sc):
    """A seeded beam, 6 undulator steps; with space charge the first half
    step is a pass of its own."""
    if sc[0] and counts == [4]:
        counts = [64]  # a single beamlet sits on its own axis: no radius
    sim = H.make_state(counts, ngrid=63, gridmax=0.3e-3, seed_power=1e6, sc=sc, longrange=bool(sc[0]))
    ctx = H.to_gpu(sim)
    _check(sim, ctx, H.steps(1, 6)[:6])
    ctx.close()


@pytest.mark.parametrize("ngrid,gridmax", [(33, 0.3e-3), (201, 0.12e-3), (251, 0.3e-3), (255, 0.06e-3)])
def test_footprints(ngrid, gridmax):
    """Footprints from a few cells to more than the tile's 3072, and grids
    that leave particles outside."""
    sim = H.make_state([2048, 512, 1300], ngrid=ngrid, gridmax=gridmax, seed_power=1e6)
    ctx = H.to_gpu(sim)
    _check(sim, ctx, H.steps(1, 4)[:4])
    ctx.close()


def test_drifts_quadrupoles_and_chicane():
    """Steps without a source between steps with one (the deposit's state
    alternates only on steps that deposit), and R56."""
    sim = H.make_state([768, 512], ngrid=63, gridmax=0.3e-3, seed_power=1e6)
    ctx = H.to_gpu(sim)
    st = list(H.steps(2, 3))
    i = next(k for k, s in enumerate(st) if s.aw == 0)
    st[i].chic_angle, st[i].chic_lb, st[i].chic_ld, st[i].chic_lt = 1e-3, 0.02, 0.01, 0.21
    _check(sim, ctx, st)
    ctx.close()


def test_harmonic_on_another_grid():
    """The harmonic's deposit shares the fundamental's scale and has its own
    footprint; its grid is smaller, so particles fall outside it only."""
    sim = H.make_state([1024, 300], ngrid=63, gridmax=0.3e-3, seed_power=1e6, timerun=False)
    sim.theta[:] += 0.2 * np.sin(3 * sim.theta)
    sim.add_harmonics([(3, 41, 0.05e-3), (2, 31, 0.2e-3)])
    rng = np.random.default_rng(1)
    for f in sim.hfields:
        f[:] = rng.normal(size=f.shape) * 1e10
    ctx = H.to_gpu(sim)
    for k, (h, ng, gm) in enumerate([(3, 41, 0.05e-3), (2, 31, 0.2e-3)]):
        ctx.add_harmonic(h, ng, gm)
        ctx.upload_harmonic(k, sim.hfields[k])
    _check(sim, ctx, H.steps(1, 5)[:5])
    for k in range(2):
        e = np.max(np.abs(ctx.download_harmonic(k) - sim.hfields[k]))
        assert e <= 1e-12 * np.max(np.abs(sim.hfields[k]))
    ctx.close()


def test_matches_separate_kernels_and_is_reproducible():
    """Two runs give the same bits, and a run whose steps are split calls
    (the separate kernels) the same field and beam to rounding."""
    st = H.steps(1, 12)[:12]
    out = []
    for mode in ("run", "run", "calls"):
        sim = H.make_state([1024, 1536, 256, 700], ngrid=63, gridmax=0.3e-3, longrange=True,
                           sc=(1, 0, 100, 0.0), seed_power=1e4)
        ctx = H.to_gpu(sim)
        gs = H.gsteps(st)
        if mode == "run":
            ctx.run(gs, cases.GAMMA0, record=("power",))
        else:
            for s in gs:
                ctx.beam_track(s, cases.GAMMA0, s.dz)
                ctx.field_track(s, s.dz)
                ctx.slippage(s.slip)
        out.append((ctx.download_beam(), ctx.download_field()[0]))
        ctx.close()
    for k in BEAM:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k
        assert np.max(np.abs(out[0][0][k] - out[2][0][k])) <= 1e-12 * np.max(np.abs(out[2][0][k])), k
    assert np.array_equal(out[0][1], out[1][1])
    assert np.max(np.abs(out[0][1] - out[2][1])) <= 1e-12 * np.max(np.abs(out[2][1]))


def test_one4one_records_across_sorts():
    """Records before and after a sort use the slices they were taken of."""
    st = list(H.steps(1, 12)[:12])
    sim = H.make_state([0, 900, 1000, 1100, 0], ngrid=41, gridmax=0.3e-3, nbins=1, shotnoise_seed=7)
    rng = np.random.default_rng(3)
    sim.theta[:] = rng.uniform(-0.5, 2 * np.pi + 0.5, len(sim.theta))
    ctx = H.to_gpu(sim)
    ctx.set_sorting(True)
    ref = H.to_gpu(sim)
    ref.set_sorting(True)
    for i, s in enumerate(st):
        s.marker = 4 if i % 5 == 3 else 0
    keys = ("power", "bunching", "energy", "xsize")
    a = ctx.run(H.gsteps(st), cases.GAMMA0, record=keys)
    for i, s in enumerate(H.gsteps(st)):
        ref.step(s, cases.GAMMA0)
        d = ref.diag()
        for k in keys:
            assert H.rel_err(a[k][i + 1], d[k]) < 1e-12, (k, i)
    assert np.array_equal(ctx.slices()[0], ref.slices()[0])
    ctx.close()
    ref.close()


def test_slow_particle_leaving_the_grid():
    """A slow particle that crosses the axis at the push and is 100 m away
    after the second half step, in a strong gradient: sqrt(faw2) / gamma is a
    million times the others' there, but it deposits nothing, so it takes
    nothing from the resolution of the others' fixed-point sums."""
    st = H.steps(1, 2)[:1]
    s = st[0]
    s.kx = s.ky = s.gradx = s.ax = s.ay = s.qf = 0.0
    s.grady = 1e3
    sim = H.make_state([1024, 512, 256], ngrid=63, gridmax=0.3e-3, timerun=False)
    sim.theta[:] += 0.3 * np.sin(sim.theta)
    sim.y *= 0.1
    gamma, gz = 4.0, 2.6e-4
    py = np.sqrt(gamma ** 2 - 1 - s.aw ** 2 - gz ** 2)
    gz = np.sqrt(gamma * gamma - 1 - s.aw * s.aw - py * py)
    for i in (5, 1030):
        sim.gamma[i], sim.px[i], sim.py[i], sim.x[i] = gamma, 0.0, py, 0.0
        sim.y[i] = -py * (0.5 * s.dz) / gz - 2e-4
    ctx = H.to_gpu(sim)
    ctx.run(H.gsteps(st), cases.GAMMA0, record=())
    sim.run(st, cases.GAMMA0, record=("power",))
    far = sim.y[[5, 1030]]
    assert np.all(np.isfinite(sim.gamma[[5, 1030]])) and np.all(far > 50), far
    f, _ = ctx.download_field()
    e = np.max(np.abs(f - sim.field)) / np.max(np.abs(sim.field))
    print(f"  field of the other particles: {e:.2e}", flush=True)
    assert e < 1e-12
    ctx.close()


@pytest.mark.parametrize("counts,value,passes", [
    ([256] * 10, -1, "split"), ([256] * 10, 1, "fused"), ([256] * 10, 0, "separate"),
    ([64] * 256, -1, "fused"), ([64] * 256, 0, "separate")])
def test_particle_passes_by_request(counts, value, passes):
    """fp64_fused 0 runs the separate kernels on any window: a record's beam
    sums are then k_diag_beam's bits, which g4mi_diag gives for the same
    particles."""
    st = H.steps(1, 2)[:2]
    sim = H.make_state(counts, ngrid=41, gridmax=0.3e-3, seed_power=1e6)
    ctx = H.to_gpu(sim)
    ctx.set_schedule("fp64_fused", value)
    assert ctx.schedule()["particle_passes"] == passes
    keys = ("bunching", "energy", "xsize", "ysize")
    g = ctx.run(H.gsteps(st), cases.GAMMA0, record=keys)
    d = ctx.diag()
    for k in keys:
        if passes == "separate":
            assert np.array_equal(g[k][-1], d[k]), k
        else:
            assert H.rel_err(g[k][-1], d[k]) < 1e-10, k
    ctx.close()


def test_separate_kernels_on_a_wide_window_with_a_harmonic():
    """256 slices with a harmonic field run the separate kernels by
    themselves: against the oracle, and the same bits twice."""
    out = []
    for _ in range(2):
        sim = H.make_state([64, 0, 132, 64] * 64, ngrid=31, gridmax=0.3e-3, seed_power=1e6, timerun=False)
        sim.theta[:] += 0.2 * np.sin(3 * sim.theta)
        sim.add_harmonics([(3, 33, 0.25e-3)])
        sim.hfields[0][:] = np.random.default_rng(2).normal(size=sim.hfields[0].shape) * 1e10
        ctx = H.to_gpu(sim)
        ctx.add_harmonic(3, 33, 0.25e-3)
        ctx.upload_harmonic(0, sim.hfields[0])
        assert ctx.schedule()["particle_passes"] == "separate"
        _check(sim, ctx, H.steps(1, 4)[:4])
        h = ctx.download_harmonic(0)
        assert np.max(np.abs(h - sim.hfields[0])) <= 1e-12 * np.max(np.abs(sim.hfields[0]))
        out.append((ctx.download_beam(), ctx.download_field()[0], h))
        ctx.close()
    for k in BEAM:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])
