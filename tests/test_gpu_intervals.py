"""Solution intervals run together (one rotate and one inversion for a group of them): every route
against the oracle on the same slices, and against calls of one interval each.

Bars: FP64 calibrations within 1e-9 rad of the oracle, mixed precision within 1e-5 (the bars of the
batched routes).  Against single-interval calls: the same sums, with the rows of a baseline split
differently over waves or chunks, so 1e-10 rad; mixed precision 1e-7, the rounding of its GEMM.
"""
import ctypes

import numpy as np
import pytest

import np_restatement as npr

pytestmark = pytest.mark.gpu

ROUTES = {
    "plain": (dict(), 40, 5),
    "wave": (dict(strategy=1), 40, 5),
    "nufft-w16": (dict(strategy=1), 130, 17),
    "mixed-wave": (dict(strategy=1, precision=1), 40, 150),  # two intervals a GEMM at most
    "mixed-nufft": (dict(strategy=1, precision=1), 130, 17),
    "tile": (dict(strategy=1, direction_block=64, direct_cube=1, channel_sum=1), 40, 5),  # one by one
    "all-pols": (dict(strategy=1, all_pols=1), 40, 5),                                     # one by one
}


def _set(leap, C, D, seed):
    s = leap.SynthMS(n_antennas=14, n_timesteps=11, n_channels=C, nan_fraction=0.002, seed=seed)
    s.fill_host(np.complex64)
    ms = s.host_dict()
    rng = np.random.default_rng(seed)
    return ms, np.asarray(ms["phase_centre"]) + rng.uniform(-0.02, 0.02, (D, 2))


@pytest.mark.parametrize("where", ["host", "device", "graph"])
@pytest.mark.parametrize("interval", [1, 3, 5])
@pytest.mark.parametrize("route", list(ROUTES))
def test_grouped_intervals(leap, ctx, oracle, route, interval, where):
    kw, C, D = ROUTES[route]
    ms, dirs = _set(leap, C, D, C + interval)
    mixed = kw.get("precision") == 1
    print(f"intervals of {interval}: {route}, {where}", flush=True)
    held = []
    if where == "host":
        view = leap.view_from_arrays(ms)
    else:
        for a in (ms["vis"], ms["uvw"]):
            held.append(ctx.malloc(a.nbytes))
            ctx.h2d(held[-1], np.ascontiguousarray(a))
        view = leap.view_from_arrays(ms, vis_device=held[0], uvw_device=held[1], vis_dtype=leap.LEAP_VIS_C64)
    try:
        md = ctx.metadata(view)
        opts = leap.options(graph=1 if where == "graph" else 0, **kw)
        want, epochs = oracle.calibrate(ms, dirs, (0, interval, -1))
        for _ in range(3 if where == "graph" else 1):
            got, at = ctx.calibrate(view, dirs, (0, interval, -1), opts=opts, md=md)
            assert np.array_equal(at, epochs)
            assert np.abs(npr.wrap(got - want)).max() < (1e-5 if mixed else 1e-9)
        if where != "device":
            return
        nbl = ms["num_baselines"]
        for s in range(len(want)):  # the same rows as a set of one interval
            rows = slice(s * interval * nbl, (s + 1) * interval * nbl)
            one = dict(ms, vis=ms["vis"][rows], uvw=ms["uvw"][rows], time=ms["time"][rows], num_rows=interval * nbl)
            alone, _ = ctx.calibrate(leap.view_from_arrays(one), dirs, (0, interval, -1),
                                     opts=leap.options(**kw), md=md)
            assert np.abs(npr.wrap(got[s] - alone[0])).max() < (1e-7 if mixed else 1e-10)
    finally:
        for p in held:
            ctx.free(p)


def test_callback_stops_between_grouped_intervals(leap, ctx):
    """A callback that asks to stop ends the call there, whatever else its group computed."""
    ms, dirs = _set(leap, 40, 3, 5)
    view = leap.view_from_arrays(ms)
    md = ctx.metadata(view)
    seen = []

    def cb(_user, sol):
        seen.append(sol.contents.index)
        return 1 if len(seen) == 2 else 0

    d = np.ascontiguousarray(dirs)
    rc = leap.lib().leap_hip_calibrate_md(ctx.h, md.h, ctypes.byref(view), d.ctypes.data_as(leap._dp), len(d), 0, 1, -1,
                                          ctypes.byref(leap.options()), leap.SOLUTION_CB(cb), None)
    assert rc == -6 and seen == [0, 1]


@pytest.mark.parametrize("route", ["plain", "wave", "mixed-wave", "nufft-w16"])
def test_slice_past_the_last_row_delivers_its_whole_intervals(leap, ctx, route):
    """Eleven timesteps in intervals of three to an end of 30: three solutions, then the range error,
    whatever the intervals are grouped into; and four of a slice that ends inside a group."""
    kw, C, D = ROUTES[route]
    ms, dirs = _set(leap, C, D, 7)
    view = leap.view_from_arrays(ms)
    md = ctx.metadata(view)
    want, _ = ctx.calibrate(view, dirs, (0, 3, -1), opts=leap.options(**kw), md=md)
    seen = []

    def cb(_user, sol):
        n = sol.contents.n_directions * sol.contents.n_antennas
        seen.append(np.ctypeslib.as_array(sol.contents.calibrations, shape=(n,)).copy())
        return 0

    d = np.ascontiguousarray(dirs)
    rc = leap.lib().leap_hip_calibrate_md(ctx.h, md.h, ctypes.byref(view), d.ctypes.data_as(leap._dp), len(d), 0, 3, 30,
                                          ctypes.byref(leap.options(**kw)), leap.SOLUTION_CB(cb), None)
    assert rc == -2 and len(seen) == len(want) == 3
    assert np.abs(npr.wrap(np.array(seen).reshape(want.shape) - want)).max() < 1e-9
    part, _ = ctx.calibrate(view, dirs, (0, 1, 4), opts=leap.options(**kw), md=md)
    every, _ = ctx.calibrate(view, dirs, (0, 1, -1), opts=leap.options(**kw), md=md)
    assert len(part) == 4 and np.abs(npr.wrap(part - every[:4])).max() < (1e-7 if kw.get("precision") else 1e-10)


@pytest.mark.parametrize("tile,D", [((64, 1), 5), ((128, 2), 70), ((256, 4), 130)])
def test_grouped_intervals_of_packed_tiles(leap, ctx, oracle, tile, D):
    """Every packed tile over several intervals at once and over one, against the oracle and each other."""
    print(f"packed tile {tile}, {D} directions", flush=True)
    ms, dirs = _set(leap, 21, D, D)
    view = leap.view_from_arrays(ms)
    md = ctx.metadata(view)
    opts = leap.options(strategy=1, channel_sum=1, direction_block=tile[0], lane_directions=tile[1])
    got, _ = ctx.calibrate(view, dirs, (0, 2, -1), opts=opts, md=md)
    want, _ = oracle.calibrate(ms, dirs[:: max(1, D // 5)], (0, 2, -1))
    assert np.abs(npr.wrap(got[:, :: max(1, D // 5)] - want)).max() < 1e-9
    rows = slice(0, 2 * ms["num_baselines"])
    one = dict(ms, vis=ms["vis"][rows], uvw=ms["uvw"][rows], time=ms["time"][rows], num_rows=rows.stop)
    alone, _ = ctx.calibrate(leap.view_from_arrays(one), dirs, (0, 2, -1), opts=opts, md=md)
    assert np.abs(npr.wrap(got[0] - alone[0])).max() < 1e-10
