"""The wave-at-a-time rotate/average: its tiles (one to four directions a lane, direction blocks
that are not full), rows of several baselines and of several timesteps, channel blocks that are
partial, odd or single, and every cube type, against the oracle (avgData within 1e-12 of its
largest magnitude, the bar of the other FP64 batched routes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def on_device(leap, ctx):
    """The set's cube and uvw on the device, freed after the test."""
    held = []

    def make(ms):
        vis = np.ascontiguousarray(ms["vis"])
        vp, up = ctx.malloc(vis.nbytes), ctx.malloc(ms["uvw"].nbytes)
        held.extend((vp, up))
        ctx.h2d(vp, vis)
        ctx.h2d(up, np.ascontiguousarray(ms["uvw"]))
        return leap.view_from_arrays(ms, vis_device=vp, uvw_device=up,
                                     vis_dtype=leap.LEAP_VIS_C64 if vis.dtype == np.complex64 else leap.LEAP_VIS_C128)

    yield make
    for p in held:
        ctx.free(p)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n_ant,T,C,P,D", [
    (4, 1, 1, 1, 1),       # one sample per baseline
    (7, 3, 33, 2, 8),      # several timesteps of a baseline, a channel past two blocks
    (40, 17, 9, 3, 9),     # a baseline's timesteps over four waves
    (91, 1, 31, 4, 16),    # 4186 baselines of one timestep: four baselines a wave
    (91, 2, 70, 1, 30),    # two directions a lane, two chunks
    (91, 3, 65, 4, 64),    # four directions a lane, a block and one channel
    (65, 2, 150, 2, 130),  # three blocks of three directions a lane
    (91, 2, 40, 4, 100),   # two blocks of 50
    (91, 1, 24, 2, 250),   # four blocks
    (91, 1, 20, 1, 300),   # five blocks of 60
])
def test_wave_horner_edges(leap, ctx, oracle, on_device, dtype, n_ant, T, C, P, D):
    print(f"wave Horner: {n_ant} antennas, {T} t, {C} ch, {P} pols, {D} directions, {np.dtype(dtype).name}", flush=True)
    s = leap.SynthMS(n_antennas=n_ant, n_timesteps=T, n_channels=C, n_pols=P, nan_fraction=0.003, seed=C + D)
    s.fill_host(dtype)
    ms = s.host_dict()
    view = on_device(ms)
    md, omd = ctx.metadata(view), oracle.metadata(ms)
    rng = np.random.default_rng(D)
    dirs = np.asarray(ms["phase_centre"]) + rng.uniform(-0.03, 0.03, (D, 2))
    got = md.rotate(view, dirs, opts=leap.options(strategy=1, channel_sum=1, direct_cube=1))
    assert ctx.last_route() == (1, 1)
    for d in sorted({0, D // 2, D - 1}):
        want = omd.rotate(dirs[d])
        assert np.abs(got[d, :, 0] - want[:, 0]).max() <= 1e-12 * np.abs(want[:, 0]).max(), d
    assert not got[:, :, 1:].any()


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n_ant,T,C,P,D", [
    (5, 1, 1, 1, 1),     # one channel: the derivative is zero
    (7, 3, 33, 2, 9),    # a channel past two blocks
    (9, 5, 70, 3, 16),   # timesteps past the four waves' rows
    (12, 2, 130, 4, 17), # direction blocks that are not full
    (12, 1, 9, 4, 256),  # the most directions
])
def test_wave_row_sums_edges(leap, ctx, oracle, on_device, dtype, n_ant, T, C, P, D):
    """The residual loss and its gradient from the row sums, and the loss alone, against the oracle
    at the bars of the other gradient tests (loss 1e-11 relative, gradients 1e-7 of the largest)."""
    print(f"row sums: {n_ant} antennas, {T} t, {C} ch, {P} pols, {D} directions, {np.dtype(dtype).name}", flush=True)
    s = leap.SynthMS(n_antennas=n_ant, n_timesteps=T, n_channels=C, n_pols=P, nan_fraction=0.003, seed=C + D)
    s.fill_host(dtype)
    ms = s.host_dict()
    view = on_device(ms)
    md = ctx.metadata(view)
    rng = np.random.default_rng(D)
    dirs = np.asarray(ms["phase_centre"]) + rng.uniform(-0.02, 0.02, (D, 2))
    off, dp = rng.normal(0, 1e-4, (D, 2)), rng.normal(0, 0.01, (n_ant, 3))
    want, want_off, want_ant = oracle.loss_grad(ms, dirs, s.enu_to_uvw, off, dp)
    ctx.set_adjoint_mode(2)
    try:
        loss, g_off, g_ant = md.loss_grad(view, dirs, s.enu_to_uvw, off, dp)
    finally:
        ctx.set_adjoint_mode(0)
    alone, _, _ = md.loss_grad(view, dirs, s.enu_to_uvw, off, dp, want_grad=False)
    assert abs(loss - want) <= 1e-11 * abs(want)
    assert abs(alone - want) <= 1e-11 * abs(want)
    assert np.abs(g_off - want_off).max() <= 1e-7 * np.abs(want_off).max()
    assert np.abs(g_ant - want_ant).max() <= 1e-7 * np.abs(want_ant).max()


@pytest.mark.parametrize("n_ant,T,P,D,precision,route", [
    (64, 1, 4, 32, 0, 1),    # 2080 rows
    (64, 1, 4, 33, 0, 4),
    (63, 1, 4, 32, 0, 4),    # 2016 rows
    (130, 2, 2, 48, 0, 1),   # 17030 rows
    (130, 2, 2, 49, 0, 4),
    (90, 4, 1, 48, 0, 4),    # 16380 rows
    (64, 1, 3, 16, 0, 1),    # a pol count the NUFFT packs
    (64, 1, 4, 32, 1, 2),    # mixed precision keeps its NUFFT
])
def test_automatic_route_of_device_cubes(leap, ctx, on_device, n_ant, T, P, D, precision, route):
    """The automatic channel sums at the borders of the rule, as close to the other route's as the
    routes of forced calls are (1e-12 of the largest magnitude in FP64, 1e-5 mixed)."""
    print(f"automatic route: {n_ant} antennas, {T} t, {P} pols, {D} directions", flush=True)
    s = leap.SynthMS(n_antennas=n_ant, n_timesteps=T, n_channels=96, n_pols=P, nan_fraction=0.003, seed=D)
    s.fill_host(np.complex64)
    ms = s.host_dict()
    view = on_device(ms)
    md = ctx.metadata(view)
    dirs = np.asarray(ms["phase_centre"]) + np.random.default_rng(D).uniform(-0.03, 0.03, (D, 2))
    got = md.rotate(view, dirs, opts=leap.options(strategy=1, precision=precision))
    assert ctx.last_route()[0] == route
    other = md.rotate(view, dirs, opts=leap.options(strategy=1, precision=precision,
                                                    channel_sum=1 if route != 1 else 4))
    bar = 1e-5 if precision else 1e-12
    assert np.abs(got[:, :, 0] - other[:, :, 0]).max() <= bar * np.abs(other[:, :, 0]).max()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_multi_set_launches_of_their_own(leap, ctx, on_device, precision):
    """A multi-set call whose sets take every kind of launch (folded sums of their own, the shared Horner
    tiles, a NUFFT group of one set) over uneven numbers of solutions: as the sets' own calls give
    (1e-9 rad in FP64, 1e-6 mixed), and the captured call and its replay equal to the eager one."""
    print(f"multi-set launches, precision {precision}", flush=True)
    sets = []
    for n_ant, T, C, D, slice_ in ((130, 3, 20, 9, (0, 1, -1)), (9, 4, 30, 5, (0, 2, -1)),
                                   (20, 4, 128, 40, (0, -1, -1)), (95, 2, 33, 70, (0, -1, -1))):
        s = leap.SynthMS(n_antennas=n_ant, n_timesteps=T, n_channels=C, nan_fraction=0.003, seed=C)
        s.fill_host(np.complex64)
        ms = s.host_dict()
        view = on_device(ms)
        dirs = np.asarray(ms["phase_centre"]) + np.random.default_rng(D).uniform(-0.02, 0.02, (D, 2))
        sets.append((ctx.metadata(view), view, dirs, slice_))
    opts = dict(strategy=1, precision=precision)
    eager = ctx.calibrate_batch(sets, leap.options(**opts))
    for (md, view, dirs, slice_), (got, epochs) in zip(sets, eager):
        want, want_epochs = ctx.calibrate(view, dirs, slice_, opts=leap.options(**opts), md=md)
        assert np.array_equal(epochs, want_epochs)
        diff = np.angle(np.exp(1j * (got - want)))
        assert np.abs(diff).max() <= (1e-6 if precision else 1e-9)
    for _ in range(3):
        again = ctx.calibrate_batch(sets, leap.options(graph=1, **opts))
        for (got, _), (want, _) in zip(again, eager):
            assert np.array_equal(got, want)


@pytest.mark.parametrize("graph", [0, 1])
def test_multi_set_calls_take_the_folded_kernel_or_the_nufft(leap, on_device, graph):
    """An FP64 set of 2,080 rows that the automatic rule gives the folded sums gets a launch of that kernel
    (its own call's bits), not a place among the shared Horner tiles, which would be tuned first; with a
    grid named it keeps the width-16 NUFFT, and so does one of 1,953 rows."""
    c = leap.Context(0)
    try:
        sets = []
        for n_ant in (64, 62):
            s = leap.SynthMS(n_antennas=n_ant, n_timesteps=1, n_channels=128, nan_fraction=0.003, seed=n_ant)
            s.fill_host(np.complex64)
            ms = s.host_dict()
            view = on_device(ms)
            dirs = np.asarray(ms["phase_centre"]) + np.random.default_rng(n_ant).uniform(-0.02, 0.02, (24, 2))
            sets.append((c.metadata(view), view, dirs, (0, -1, -1)))
        opts = dict(strategy=1, graph=graph)
        for case, route in (([sets[0]], 1), (sets, 4), ([sets[1]], 4)):
            got = c.calibrate_batch(case, leap.options(**opts))
            assert c.last_route()[0] == route and c.last_direction_block() == 0
            for (md, view, dirs, slice_), (cal, _) in zip(case, got):
                want, _ = c.calibrate(view, dirs, slice_, opts=leap.options(strategy=1), md=md)
                assert np.abs(np.angle(np.exp(1j * (cal - want)))).max() <= (0 if md is sets[0][0] else 1e-9)
        named = c.calibrate_batch(sets, leap.options(workgroups_per_cu=4, **opts))
        assert c.last_route()[0] == 4 and c.last_direction_block() == 0
        for (cal, _), (want, _) in zip(named, c.calibrate_batch(sets, leap.options(**opts))):
            assert np.abs(np.angle(np.exp(1j * (cal - want)))).max() <= 1e-9
    finally:
        c.close()
