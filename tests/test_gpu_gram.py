"""The device pseudo-inverse (block sweeps of 32 antennas) around its tile edges.

Against the host routine leap_phase_matrix_pinv, an unblocked Cholesky of the same
exact integer matrix.  Both invert a diagonally dominant matrix and add the exact ones
of the constraint's component, with N rounded steps per entry each: the tolerance is
16 N eps of the largest entry.
"""
import ctypes

import numpy as np
import pytest

import np_restatement as npr

pytestmark = pytest.mark.gpu


def _ms(a1, a2, fg):
    nbl, n_ant = len(a1), int(max(a1.max(), a2.max())) + 1
    return {"num_stations": n_ant, "total_antennas": n_ant, "num_baselines": nbl, "num_rows": nbl, "num_channels": 1,
            "num_pols": 1, "freq_start_hz": 1e8, "freq_inc_hz": 1e6, "phase_centre": (0.1, -0.5), "antenna1": a1,
            "antenna2": a2, "time": np.zeros(nbl), "flag": fg, "uvw": np.zeros((nbl, 3)),
            "vis": np.zeros((nbl, 1, 1), dtype=np.complex128)}


@pytest.mark.parametrize("graph", ["dense", "chain", "split"])
@pytest.mark.parametrize("n_ant", [2, 31, 32, 33, 64, 65, 130])
def test_pseudo_inverse_at_tile_edges(leap, ctx, n_ant, graph):
    """dense: 3% flagged; chain: only neighbours, repeated twice (the longest paths and twice the
    counts); split: two halves, one without the constraint, and one antenna without baselines."""
    from test_capi import _host_phase_matrix

    a1, a2 = (x.astype(np.int32) for x in np.triu_indices(n_ant))
    rng = np.random.default_rng(n_ant)
    fg = np.zeros(len(a1), dtype=np.uint8)
    if graph == "dense":
        fg[n_ant:] = rng.random(len(a1) - n_ant) < 0.03
    elif graph == "chain":
        fg[:] = a2 - a1 != 1
        fg[0] = 0
        a1, a2, fg = np.tile(a1, 2), np.tile(a2, 2), np.tile(fg, 2)
    else:
        half = n_ant // 2
        fg[:] = ((a1 < half) != (a2 < half)) | ((a2 == n_ant - 1) & (n_ant > 2))
        fg[0] = 0
    print(f"pseudo-inverse: {n_ant} antennas, {graph}", flush=True)
    got = ctx.metadata(leap.view_from_arrays(_ms(a1, a2, fg)), ref_ant=0).copy()
    for name, ref in (("", None), ("1", 0)):
        A, _, want = _host_phase_matrix(leap, a1, a2, fg, ref)
        assert np.array_equal(got["A" + name], A)
        scale = max(1.0, np.abs(want).max())
        err = np.abs(got["Ad" + name] - want).max() / scale
        print(f"Ad{name}: {err:.2e}")
        assert err <= 16 * n_ant * np.finfo(float).eps


@pytest.mark.parametrize("n_dirs", [1, 5])
@pytest.mark.parametrize("n_ant,graph", [(2, "dense"), (63, "dense"), (64, "split"), (65, "dense"), (130, "split")])
def test_inversion_through_antenna_sums(leap, ctx, n_ant, graph, n_dirs):
    """cal = Ad dphi + Ad1 phi1 of random averages against LAPACK's pseudo-inverses (the 1e-9 rad bar of
    the calibrations), around the kernels' 64-antenna blocks, with components without the constraint,
    and with the pseudo-inverse taken from the context's cache the second time."""
    a1, a2 = (x.astype(np.int32) for x in np.triu_indices(n_ant))
    rng = np.random.default_rng(10 * n_ant + n_dirs)
    fg = np.zeros(len(a1), dtype=np.uint8)
    if graph == "split":
        fg[:] = ((a1 < n_ant // 2) != (a2 < n_ant // 2)) | (a2 == n_ant - 1)
        fg[0] = 0
    print(f"inversion: {n_ant} antennas, {graph}, {n_dirs} directions", flush=True)
    avg = rng.normal(size=(n_dirs, len(a1), 1)) + 1j * rng.normal(size=(n_dirs, len(a1), 1))
    view = leap.view_from_arrays(_ms(a1, a2, fg))
    A, I = npr.phase_matrix(a1, a2, fg)
    A1, I1 = npr.phase_matrix(a1, a2, fg, 0)
    Ad, Ad1 = np.linalg.pinv(A), np.linalg.pinv(A1)
    want = np.array([npr.apply_inversion(x, A, I, A1, I1, Ad, Ad1) for x in avg])
    for cached in (False, True, True):
        md = ctx.metadata(view, ref_ant=0, use_cache=cached)
        assert np.abs(npr.wrap(md.apply_inversion(avg) - want)).max() < 1e-9


def test_a_metadata_keeps_no_scratch(leap, ctx):
    """Device memory of kept metadata with few baselines, where the antennas' square counts: what calls
    read (G+ with and without the ones for A and A1, Ad, Ad1 and Ad's BF16 planes) and a tenth, without the
    two more matrices each that the inversion works in."""
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    n, count = 1024, 5
    a1 = np.concatenate([np.arange(n - 1), [0]]).astype(np.int32)
    a2 = np.concatenate([np.arange(1, n), [n - 1]]).astype(np.int32)
    view = leap.view_from_arrays(_ms(a1, a2, np.zeros(n, dtype=np.uint8)))
    kept = [ctx.metadata(view, ref_ant=0)]  # the context's own buffers are there after the first
    K, K1 = kept[0].K, kept[0].K1
    before = free_bytes()
    kept += [ctx.metadata(view, ref_ant=0) for _ in range(count)]
    used = (before - free_bytes()) / count
    need = 8 * (4 * n * n + (K + K1) * n) + 6 * (K + 31) // 32 * 32 * n
    print(f"{used / 2**20:.1f} MiB a metadata, {need / 2**20:.1f} read by calls", flush=True)
    assert used <= 1.1 * need + 4 * 2**20
