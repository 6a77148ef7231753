"""Host-resident visibilities: staged through the pinned double buffer (every
path) or packed to pol 0 on the host (the packed path).

The device receives the same values either way, so results equal those of the
same cube resident on the device bit for bit; the packed path sends only pol 0
(a quarter of a 4-pol cube) across the bus.  The cube is large enough to need
several pinned chunks.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dirs_near(centre, n, seed, spread=0.02):
    rng = np.random.default_rng(seed)
    return np.column_stack([centre[0] + rng.uniform(-spread, spread, n), centre[1] + rng.uniform(-spread, spread, n)])


@pytest.fixture(scope="module", params=["c64", "c128"])
def big(request, leap, ctx):
    """128 antennas (8256 baselines) x 80 t x 48 ch x 4 pols with NaNs: 1.27 GB c64 / 2.5 GB c128 on the host."""
    c64 = request.param == "c64"
    vd = leap.LEAP_VIS_C64 if c64 else leap.LEAP_VIS_C128
    dt = np.complex64 if c64 else np.complex128
    s = leap.SynthMS(n_antennas=128, n_timesteps=80, n_channels=48, nan_fraction=1e-4, seed=95)
    nbytes = s.num_rows * s.num_channels * s.num_pols * np.dtype(dt).itemsize
    vis_p = ctx.malloc(nbytes)
    uvw_p = ctx.malloc(s.num_rows * 24)
    ctx.synth_fill_device(s, vd, vis_p, uvw_p)
    host = np.empty((s.num_rows, s.num_channels, s.num_pols), dtype=dt)
    ctx.d2h(host, vis_p)
    ms = s.host_dict(host)
    dev_view = leap.view_from_arrays(ms, vis_device=vis_p, vis_dtype=vd, uvw_device=uvw_p)
    host_view = leap.view_from_arrays(ms)
    md = ctx.metadata(host_view)
    yield s, ms, md, host_view, dev_view, np.dtype(dt).itemsize
    ctx.free(vis_p)
    ctx.free(uvw_p)


# Packed cases name their tile: a tuned call on the device cube would be routed straight from the cube
# at this direction count, while a host cube always takes the packed route.
PK = dict(strategy=1, direction_block=64, lane_directions=1)


@pytest.mark.parametrize("opts_kw", [PK, dict(PK, pack_timesteps=30), dict(PK, precision=1),
                                     dict(strategy=1, direct_cube=1), dict(strategy=0)],
                         ids=["packed", "packed-chunks", "packed-mixed", "direct-cube", "per-direction"])
def test_host_cube_equals_device_cube(leap, ctx, big, opts_kw):
    s, ms, md, host_view, dev_view, elem = big
    if opts_kw.get("precision") == 1 and elem == 16:
        pytest.skip("mixed precision is run on the complex64 cube")
    dirs = dirs_near(ms["phase_centre"], 3 if opts_kw["strategy"] == 0 else 40, 6)
    opts = leap.options(**opts_kw)
    got_host, eh = ctx.calibrate(host_view, dirs, (0, 40, -1), opts=opts, md=md)
    staged = ctx.last_staged_bytes()
    got_dev, ed = ctx.calibrate(dev_view, dirs, (0, 40, -1), opts=opts, md=md)
    assert ctx.last_staged_bytes() == 0
    assert np.array_equal(got_host, got_dev) and np.array_equal(eh, ed)
    rc = s.num_rows * s.num_channels
    if opts_kw["strategy"] == 1 and not opts_kw.get("direct_cube"):
        assert staged == rc * 2 * (elem // 2)  # pol 0 only, in the source precision
    else:
        assert staged == rc * s.num_pols * elem  # whole rows


@pytest.mark.parametrize("strategy", [0, 1])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n_ant,T,C,P", [(3, 1, 1, 1), (16, 15, 125, 4), (16, 15, 129, 4), (33, 30, 70, 3), (40, 41, 64, 2)])
def test_staged_pieces(leap, ctx, dtype, strategy, n_ant, T, C, P):
    """Host cubes of one sample up to several pieces of the staging copy (8 MiB, filled in blocks of
    512 KiB), whole rows or pol 0 alone, give the bits of the same cube on the device."""
    print(f"staged pieces: {n_ant} antennas, {T} t, {C} ch, {P} pols, {np.dtype(dtype).name}", flush=True)
    s = leap.SynthMS(n_antennas=n_ant, n_timesteps=T, n_channels=C, n_pols=P, nan_fraction=0.002, seed=C)
    s.fill_host(dtype)
    ms = s.host_dict()
    vis = np.ascontiguousarray(ms["vis"])
    host_view = leap.view_from_arrays(ms)
    md = ctx.metadata(host_view)
    vis_p, uvw_p = ctx.malloc(vis.nbytes), ctx.malloc(ms["uvw"].nbytes)
    try:
        ctx.h2d(vis_p, vis)
        ctx.h2d(uvw_p, np.ascontiguousarray(ms["uvw"]))
        dev_view = leap.view_from_arrays(ms, vis_device=vis_p, uvw_device=uvw_p,
                                         vis_dtype=leap.LEAP_VIS_C64 if dtype is np.complex64 else leap.LEAP_VIS_C128)
        dirs = dirs_near(ms["phase_centre"], 3, C)
        opts = leap.options(strategy=strategy, **(dict(direction_block=64, lane_directions=1) if strategy else {}))
        got, _ = ctx.calibrate(host_view, dirs, opts=opts, md=md)
        elem = vis.itemsize // 2
        assert ctx.last_staged_bytes() == vis.size // P * 2 * elem * (1 if strategy else P)
        want, _ = ctx.calibrate(dev_view, dirs, opts=opts, md=md)
        assert np.array_equal(got, want)
    finally:
        ctx.free(vis_p)
        ctx.free(uvw_p)
