"""The per-direction FP64 rotate/average where its launch changes: directions per pass (1, 2, 4, 8
and groups that are not full), waves per baseline (16 below 512 baselines with long rows, 4, and 1
from 4096), the 32-row chunks of its shift factors, rows shorter and longer than a wave, wavelengths
past the LDS table, and samples that take the plain form (non-finite values; shifts past 2^26 rad and
non-finite uvw below).  Against the oracle, avgData within 1e-12 of its largest magnitude and calibrations
within 1e-9 rad (the bars of test_gpu_parity.py)."""
import numpy as np
import pytest

import np_restatement as npr

pytestmark = pytest.mark.gpu


def _check(leap, ctx, oracle, ms, n_dirs, seed, calibrate=True):
    rng = np.random.default_rng(seed)
    dirs = np.asarray(ms["phase_centre"]) + rng.uniform(-0.03, 0.03, (n_dirs, 2))
    view = leap.view_from_arrays(ms)
    md, omd = ctx.metadata(view), oracle.metadata(ms)
    got = md.rotate(view, dirs)
    for d in range(n_dirs):
        want = omd.rotate(dirs[d])
        assert np.abs(got[d] - want).max() <= 1e-12 * np.abs(want).max(), d
    if calibrate:
        cal, _ = ctx.calibrate(view, dirs, md=md)
        want, _ = oracle.calibrate(ms, dirs)
        assert np.abs(npr.wrap(cal - want)).max() < 1e-9


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n_ant,T,C,P,D", [
    (5, 1, 1, 1, 1),      # one sample per baseline
    (6, 33, 130, 2, 3),   # 16 waves per baseline, a second chunk of one row
    (9, 3, 7, 3, 5),      # rows shorter than a wave, 3 pols
    (12, 32, 128, 4, 8),  # a full pass of 8 directions, rows of whole waves
    (12, 2, 1030, 1, 9),  # wavelengths past the LDS table; 9 directions: two groups
    (34, 9, 75, 4, 1),    # 595 baselines, a direction or two of 4 pols: complex128 samples loaded a pol a lane
    (91, 2, 5, 4, 3),     # the same with one wave per baseline and rows shorter than its loads
    (90, 1, 5, 4, 17),    # 4095 baselines: four waves each
    (91, 1, 5, 4, 17),    # 4186 baselines: one wave each
])
def test_plain_rotate_edges(leap, ctx, oracle, dtype, n_ant, T, C, P, D):
    print(f"plain rotate: {n_ant} antennas, {T} t, {C} ch, {P} pols, {D} directions, {np.dtype(dtype).name}", flush=True)
    s = leap.SynthMS(n_antennas=n_ant, n_timesteps=T, n_channels=C, n_pols=P, nan_fraction=0.002, seed=n_ant + C)
    s.fill_host(dtype)
    _check(leap, ctx, oracle, s.host_dict(), D, 7 * C + D)


def test_plain_rotate_extreme_rows(leap, ctx, oracle):
    """Rows whose shifts pass 2^26 rad, and rows with a NaN or an infinity in uvw (every sample of
    such a row rotates to NaN and is skipped).  The dd matrices of the two sides may differ by two
    roundings of an entry, which a row of length L turns into 2 pi nu / c L eps rad a term: that times
    the sum of |v| is allowed on the baselines of the long rows, the usual bar on the others."""
    s = leap.SynthMS(n_antennas=8, n_timesteps=5, n_channels=70, seed=3)
    s.fill_host()
    ms = s.host_dict()
    nbl = ms["num_baselines"]
    ms["uvw"] = ms["uvw"].copy()
    ms["uvw"][3::17] *= 1e7
    length = np.linalg.norm(ms["uvw"], axis=1)
    ms["uvw"][5, 1] = np.nan
    ms["uvw"][11, 2] = np.inf
    size = np.abs(ms["vis"][:, :, 0]).sum(axis=1)
    nu = ms["freq_start_hz"] + 69 * ms["freq_inc_hz"]
    phase = 2 * np.pi * nu / npr.C_LIGHT * length * np.finfo(float).eps
    bar = np.zeros(nbl)
    np.add.at(bar, np.arange(len(size)) % nbl, 6 * phase * size)  # three entries, two roundings each
    dirs = np.asarray(ms["phase_centre"]) + [[0.02, -0.01], [-0.03, 0.02], [0.001, 0.03]]
    assert 2 * np.pi * nu / npr.C_LIGHT * length.max() * 1e-2 > 2 ** 26
    view = leap.view_from_arrays(ms)
    got, omd = ctx.metadata(view).rotate(view, dirs), oracle.metadata(ms)
    for d in range(len(dirs)):
        want = omd.rotate(dirs[d])
        assert np.isfinite(want).all()
        err = np.abs(got[d, :, 0] - want[:, 0])
        print(f"direction {d}: error over bar {(err / (bar + 1e-12 * np.abs(want).max())).max():.2e}")
        assert (err <= bar + 1e-12 * np.abs(want).max()).all()


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_plain_rotate_channel_at_zero_hz(leap, ctx, oracle, dtype):
    """A band through 0 Hz: that channel's wavelength is infinite and its phase zero."""
    s = leap.SynthMS(n_antennas=9, n_timesteps=2, n_channels=9, freq_start_hz=-8e6, freq_inc_hz=2e6, seed=9)
    s.fill_host(dtype)
    _check(leap, ctx, oracle, s.host_dict(), 5, 9, calibrate=False)


@pytest.mark.parametrize("opts_kw", [dict(), dict(strategy=1, channel_sum=1)], ids=["plain", "folded"])
def test_calibrations_and_times_of_small_and_large_results(leap, ctx, opts_kw):
    """Results up to 32,768 calibrations are written to pinned memory by the inversion, larger ones are
    copied: a direction's calibrations are the same (1e-9 rad) either way.  The rotate's time is that
    of one launch and lies inside the call's."""
    s = leap.SynthMS(n_antennas=20, n_timesteps=2, n_channels=3, seed=20)
    s.fill_host(np.complex64)
    ms = s.host_dict()
    vis = np.ascontiguousarray(ms["vis"])
    vp, up = ctx.malloc(vis.nbytes), ctx.malloc(ms["uvw"].nbytes)
    try:
        ctx.h2d(vp, vis)
        ctx.h2d(up, np.ascontiguousarray(ms["uvw"]))
        view = leap.view_from_arrays(ms, vis_device=vp, uvw_device=up, vis_dtype=leap.LEAP_VIS_C64)
        md = ctx.metadata(view)
        dirs = np.asarray(ms["phase_centre"]) + np.random.default_rng(20).uniform(-0.02, 0.02, (1639, 2))
        got = []
        for n in (1638, 1639):
            cal, _ = ctx.calibrate(view, dirs[:n], opts=leap.options(**opts_kw), md=md)
            got.append(cal)
            ms_rotate, launches, ms_total = ctx.last_kernel_times()
            assert launches == 1 and 0 < ms_rotate < ms_total
        assert np.abs(npr.wrap(got[0] - got[1][:, :1638])).max() < 1e-9
        ctx.calibrate(view, dirs[:3], (0, 1, -1), opts=leap.options(**opts_kw), md=md)  # two solutions, one launch
        assert ctx.last_kernel_times()[1] == 1
    finally:
        ctx.free(vp)
        ctx.free(up)


@pytest.mark.parametrize("n_ant,autos,D", [(2, 1, 1), (3, 1, 5), (45, 0, 3), (46, 0, 3), (46, 1, 2), (64, 0, 2)])
def test_inversion_of_few_antennas(leap, ctx, oracle, n_ant, autos, D):
    """Calibrations by the one-launch inversion (up to 64 antennas and 1,024 rows: 990 rows of 45 antennas)
    and, past it (1,035 rows of 46), by the three launches, with flagged baselines and NaNs, within
    1e-9 rad of the oracle (the bar of test_gpu_parity.py)."""
    print(f"inversion: {n_ant} antennas, autocorrelations {autos}, {D} directions", flush=True)
    s = leap.SynthMS(n_antennas=n_ant, autocorrelations=autos, n_timesteps=2, n_channels=3, nan_fraction=0.01,
                     flag_fraction=0.05 if n_ant > 10 else 0.0, seed=n_ant)
    s.fill_host(np.complex64)
    ms = s.host_dict()
    dirs = np.asarray(ms["phase_centre"]) + np.random.default_rng(D).uniform(-0.02, 0.02, (D, 2))
    got, _ = ctx.calibrate(leap.view_from_arrays(ms), dirs)
    want, _ = oracle.calibrate(ms, dirs)
    assert np.abs(npr.wrap(got - want)).max() < 1e-9
