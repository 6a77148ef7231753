"""The wave-at-a-time Horner rotate/average: its tiles (8 to 256 directions a wave, direction blocks
that are not full), rows of several baselines and of several timesteps, channel chunks that are
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
    (7, 3, 33, 2, 8),      # 16 rows a wave, several baselines and timesteps, chunks of 8 and 16 channels
    (40, 17, 9, 3, 9),     # a direction past a full block
    (91, 1, 31, 4, 16),    # 4186 baselines of one timestep: eight baselines a wave
    (91, 2, 70, 1, 30),    # four rows a wave, two chunks
    (91, 3, 65, 4, 64),    # two rows a wave, a chunk and one channel
    (65, 2, 150, 2, 130),  # narrow tiles (2145 baselines), 17 blocks
    (91, 2, 40, 4, 100),   # 128 directions a wave
    (91, 1, 24, 2, 250),   # four directions a lane
    (91, 1, 20, 1, 300),   # two blocks of 150
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
