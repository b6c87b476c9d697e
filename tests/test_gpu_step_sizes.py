"""The tables kept per step size (ADI factors and bands, spectral kernels)
against the oracle: a line with more distinct step sizes than a context
keeps, walked twice so that every table is dropped and built again."""
import ctypes as C

import numpy as np
import pytest

import cases
import g4mi
import harness as H
import oracle_py as O

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


@pytest.mark.parametrize("kernel", [-1, 0, 3, 4, 5])
@pytest.mark.parametrize("ngrid", [31, 32, 65, 97])
def test_harmonic_field_in_each_adi_kernel(kernel, ngrid):
    """A third-harmonic field on its own grid (at, below and above the edges
    of the 32-cell tiles and 64-column wavefronts) in the tuned and in each
    fixed ADI kernel, over three step sizes with other band widths; a kernel
    that does not take a step size falls back to the tuner's."""
    sim = H.make_state([256] * 9, ngrid=41, gridmax=0.3e-3, seed_power=1e6, timerun=False)
    # bunched at the harmonic: an unmodulated quiet beam's source is rounding noise
    sim.theta[:] += 0.2 * np.sin(3 * sim.theta)
    sim.add_harmonics([(3, ngrid, 0.25e-3)])
    rng = np.random.default_rng(ngrid)
    sim.hfields[0][:] = rng.normal(size=sim.hfields[0].shape) * 1e10
    ctx = H.to_gpu(sim)
    ctx.add_harmonic(3, ngrid, 0.25e-3)
    ctx.upload_harmonic(0, sim.hfields[0])
    ctx.set_schedule("adi_kernel", kernel)
    st = H.steps(1, 2)
    one = H.gsteps(st)[0]
    for delz in (0.015, 0.4, 0.015, 3.0):
        ctx.field_track(one, delz)
        H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
    e = np.max(np.abs(ctx.download_harmonic(0) - sim.hfields[0])) / np.max(np.abs(sim.hfields[0]))
    print(f"  harmonic {ngrid}^2, kernel {kernel}: {e:.2e}", flush=True)
    assert e < 4e-13  # four steps of the single step's 1e-13 bar
    ctx.close()


STRIP_GRIDS = [3, 5, 16, 17, 18, 26, 33, 34, 35, 42, 48, 49, 50, 51, 54, 55, 64, 100, 105, 130, 255, 300]


@pytest.mark.parametrize("delz", [0.004, 0.015, 0.03, 0.045, 0.1, 0.24, 0.55, 0.75])
@pytest.mark.parametrize("ngrid", STRIP_GRIDS)
def test_column_strips(ngrid, delz):
    """The strip kernel (adi_kernel 4) at grids narrower than its halo, at the
    edges of its strips (54 to 18 columns) and blocks of 8 rows, with the
    source's footprint anywhere in the grid (and none), for one step size per
    form (6 to 24 terms), against the oracle: two steps of the
    single step's 1e-13 bar."""
    gridmax = 0.5e-3 * (ngrid - 1) / 150  # the cell of 151 columns on 1 mm
    sim = H.make_state([256, 512, 0, 1024, 256], ngrid=ngrid, gridmax=gridmax, timerun=False)
    rng = np.random.default_rng(ngrid)
    sim.x += gridmax * 0.9 * np.repeat([0, -1, 0, 1, 0], [256, 512, 0, 1024, 256])
    sim.y += gridmax * 0.9 * np.repeat([0, 1, 0, -1, -1], [256, 512, 0, 1024, 256])
    sim.theta += 0.3 * np.sin(sim.theta)
    sim.field[:] = rng.normal(size=sim.field.shape) * 1e9
    ctx = H.to_gpu(sim)
    ctx.set_schedule("adi_kernel", 4)
    st = H.steps(1, 2)
    one = H.gsteps(st)[0]
    for _ in range(2):
        ctx.field_track(one, delz)
        H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
    assert ctx.schedule()["adi"] == "strips"
    f, _ = ctx.download_field()
    err = np.max(np.abs(f - sim.field)) / np.max(np.abs(sim.field))
    d = ctx.diag()
    w = (sim.field ** 2).sum(axis=2).sum(axis=1)
    print(f"  {ngrid}^2, delz {delz}: {err:.2e}", flush=True)
    assert err < 2e-13
    assert np.max(np.abs(d["power"] / d["power"].sum() - w / w.sum())) < 1e-12
    ctx.close()


@pytest.mark.parametrize("ngrid,delz", [(n, d) for n in STRIP_GRIDS for d in (0.004, 0.03, 0.06, 0.1, 0.24, 0.4, 0.75, 1.1)] +
                         [(5, 4.0), (9, 4.0)])
def test_column_strips_mixed(ngrid, delz):
    """The mixed form's strip kernel (mixed_adi 2) at the same edges, one step
    size per form (6 to 24 terms) and beyond them, against the oracle: without current, two
    steps of one FP32 rounding each (2^-24 of a component, so of the largest
    value) on a seed that FP32 holds exactly."""
    gridmax = 0.5e-3 * (ngrid - 1) / 150
    sim = H.make_state([256] * 3, ngrid=ngrid, gridmax=gridmax, timerun=False)
    sim.current[:] = 0.0
    rng = np.random.default_rng(ngrid)
    sim.field[:] = rng.normal(size=sim.field.shape).astype(np.float32) * 2.0 ** 30
    ctx = H.to_gpu(sim, precision=g4mi.FP32)
    ctx.set_schedule("mixed_adi", 2)
    st = H.steps(1, 2)
    st[0].dz = delz
    for _ in range(2):
        O.lib().orc_step_all(C.byref(sim.s), C.byref(st[0]), cases.GAMMA0)
        ctx.step(H.gsteps(st)[0], cases.GAMMA0)
    assert ctx.schedule()["adi"] == "strips"
    f, _ = ctx.download_field()
    err = np.max(np.abs(f - sim.field)) / np.max(np.abs(sim.field))
    d = ctx.diag()
    w = (sim.field ** 2).sum(axis=2).sum(axis=1)
    print(f"  {ngrid}^2, delz {delz}: {err:.2e}", flush=True)
    assert err < 2.5 * 2.0 ** -24
    assert np.max(np.abs(d["power"] / d["power"].sum() - w / w.sum())) < 1e-6
    ctx.close()


@pytest.mark.parametrize("delz", [0.004, 0.2, 2.0, 40.0, 300.0, 4000.0])
@pytest.mark.parametrize("ngrid", [3, 4, 31, 63, 64, 65, 128, 129, 192, 193, 256, 257, 300])
def test_lines(ngrid, delz):
    """The line kernels (adi_kernel 5) at the edges of a lane's cells (64, 128,
    192, 256 columns) and of the blocks of four columns, for step sizes whose
    convolution needs 8 terms to many times the line's length (its distances
    taken modulo the period) and one that they leave to Thomas' sweeps, against
    the oracle: two steps of the single step's 1e-13 bar, and the field sums."""
    gridmax = 0.5e-3 * (ngrid - 1) / 150
    sim = H.make_state([256, 512, 0], ngrid=ngrid, gridmax=gridmax, timerun=False)
    rng = np.random.default_rng(ngrid)
    sim.theta += 0.3 * np.sin(sim.theta)
    sim.field[:] = rng.normal(size=sim.field.shape) * 1e9
    ctx = H.to_gpu(sim)
    ctx.set_schedule("adi_kernel", 5)
    st = H.steps(1, 2)
    one = H.gsteps(st)[0]
    for _ in range(2):
        ctx.field_track(one, delz)
        H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
    assert ctx.schedule()["adi"] == ("lines" if delz < 1000 else "thomas" if ngrid > 8 else "band")
    f, _ = ctx.download_field()
    err = np.max(np.abs(f - sim.field)) / np.max(np.abs(sim.field))
    d = ctx.diag()
    w = (sim.field ** 2).sum(axis=2).sum(axis=1)
    print(f"  {ngrid}^2, delz {delz}: {err:.2e}", flush=True)
    assert err < 2e-13
    assert np.max(np.abs(d["power"] / d["power"].sum() - w / w.sum())) < 1e-12
    ctx.close()


@pytest.mark.parametrize("delz", [0.015, 0.4, 2.0])
@pytest.mark.parametrize("ngrid", [31, 151, 255])
def test_thomas_by_request(ngrid, delz):
    """adi_kernel 0 runs the reference's recurrence, for the fundamental and a
    harmonic field, whatever other kernels hold the step size: its fields
    differ from the lines' by rounding, not by nothing."""
    out = []
    for kernel in (0, 5):
        sim = H.make_state([256] * 2, ngrid=ngrid, gridmax=0.5e-3 * (ngrid - 1) / 150, timerun=False)
        sim.theta[:] += 0.2 * np.sin(3 * sim.theta)
        sim.add_harmonics([(3, ngrid, sim.s.gridmax)])
        rng = np.random.default_rng(ngrid)
        for f in (sim.field, sim.hfields[0]):
            f[:] = rng.normal(size=f.shape) * 1e10
        ctx = H.to_gpu(sim)
        ctx.add_harmonic(3, ngrid, sim.s.gridmax)
        ctx.upload_harmonic(0, sim.hfields[0])
        ctx.set_schedule("adi_kernel", kernel)
        st = H.steps(1, 2)
        ctx.field_track(H.gsteps(st)[0], delz)
        H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
        assert ctx.schedule()["adi"] == ("thomas" if kernel == 0 else "lines")
        got = (ctx.download_field()[0], ctx.download_harmonic(0))
        d = ctx.diag()
        ctx.close()
        for f, ref in zip(got, (sim.field, sim.hfields[0])):
            assert np.max(np.abs(f - ref)) < 1e-13 * np.max(np.abs(ref))
        w = (sim.field ** 2).sum(axis=2).sum(axis=1)
        assert np.max(np.abs(d["power"] / d["power"].sum() - w / w.sum())) < 1e-12
        out.append(got)
    for a, b in zip(*out):
        assert not np.array_equal(a, b)


@pytest.mark.parametrize("kernel", [1, 2, 3, 4])
def test_request_between_steps_of_one_size(kernel):
    """A kernel asked for between two steps of a size that it does not hold
    leaves the tuner's choice there (with and without a harmonic field), and
    is taken at the next step size that it does hold."""
    sim = H.make_state([256] * 4, ngrid=151, seed_power=1e6, timerun=False)
    # bunched at the harmonic: an unmodulated quiet beam's source is rounding noise
    sim.theta[:] += 0.2 * np.sin(3 * sim.theta)
    sim.add_harmonics([(3, 151, sim.s.gridmax)])
    sim.hfields[0][:] = np.random.default_rng(kernel).normal(size=sim.hfields[0].shape) * 1e10
    ctx = H.to_gpu(sim)
    ctx.add_harmonic(3, 151, sim.s.gridmax)
    ctx.upload_harmonic(0, sim.hfields[0])
    st = H.steps(1, 2)
    one = H.gsteps(st)[0]
    for k, delz in enumerate((5.0, 5.0, 0.015)):
        ctx.field_track(one, delz)
        H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
        if k == 0:
            ctx.set_schedule("adi_kernel", kernel)
        else:
            assert (ctx.schedule()["adi_kernel"] == kernel) == (delz == 0.015)
        f, _ = ctx.download_field()
        assert np.max(np.abs(f - sim.field)) < 1e-13 * 3 * np.max(np.abs(sim.field)), k
        e = np.max(np.abs(ctx.download_harmonic(0) - sim.hfields[0])) / np.max(np.abs(sim.hfields[0]))
        assert e < 4e-13
    ctx.close()


def test_step_size_that_is_no_number():
    """A step of NaN gives the oracle's NaN field, whatever step sizes came
    before it, and leaves their choices alone."""
    sim = H.make_state([256] * 3, ngrid=65, seed_power=1e6, timerun=False)
    ctx = H.to_gpu(sim)
    one = H.gsteps(H.steps(1, 2))[0]
    for kernel in (-1, 3, 4):
        ctx.set_schedule("adi_kernel", kernel)
        ctx.upload_field(sim.field, 0)
        for delz in (0.015, 0.03):
            ctx.field_track(one, delz)
        before = ctx.schedule()["adi_by_delz"]
        ctx.field_track(one, float("nan"))
        assert np.all(np.isnan(ctx.download_field()[0]))
        assert ctx.schedule()["adi_by_delz"] == before
    ctx.close()


@pytest.mark.parametrize("ngrid,ns,delz,kernels", [
    (151, 2, 0.015, ("band", "strips")), (61, 511, 0.015, ("band", "strips")), (61, 512, 0.015, ("strips",)),
    (151, 2, 0.2, ("lines",)), (61, 255, 0.2, ("lines",)), (61, 256, 0.2, ("strips",)),
    (151, 2, 5.0, ("lines",)), (31, 1024, 5.0, ("lines",)), (151, 2, 4000.0, ("thomas",)),
    (521, 2, 0.2, ("band", "strips")), (521, 2, 0.6, ("strips",)), (521, 2, 5.0, ("thomas",))])
def test_choice_of_kernel(ngrid, ns, delz, kernels):
    """The rule on both sides of its lines (8 columns of the band, half a strip
    and one strip per SIMD, the strips' and the lines' step sizes, grids of
    512), and the kernel chosen against the oracle."""
    sim = H.make_state([4] * ns, ngrid=ngrid, gridmax=0.5e-3 * (ngrid - 1) / 150, timerun=False)
    sim.field[:] = np.random.default_rng(ns).normal(size=sim.field.shape) * 1e9
    ctx = H.to_gpu(sim)
    st = H.steps(1, 2)
    st[0].aw = 0
    ctx.field_track(H.gsteps(st)[0], delz)
    sch = ctx.schedule()
    assert sch["adi"] in kernels, sch
    assert sum(m > 0 for m in sch["adi_tuned_ms"]) == (2 if len(kernels) == 2 else 0)
    H.oracle_call("orc_field_advance", sim, C.byref(st[0]), C.c_double(delz))
    f, _ = ctx.download_field()
    assert np.max(np.abs(f - sim.field)) < 1e-13 * np.max(np.abs(sim.field))
    ctx.close()
