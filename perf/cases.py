"""Performance cases of the calibrator: what a user's program has it do, over the real range of sizes.

Every case is a synthetic measurement set (point sources under per-antenna phase screens, plus noise)
and calls of the Python binding's public entry points: `Context.calibrate`, `Context.calibrate_batch`
and `leap_torch.residual_loss` with its backward pass.  The sizes are those of the benchmark, the tests
and the command line's defaults, and odd ones between them.  `draw` gives more of the same ranges.

Fields of a case:
  kind        "calibrate", "sets" (several uneven measurement sets in one call) or "grad" (loss + gradients)
  array       "disk" (1.5 km, 169.6 MHz, 40 kHz channels) or "spiral" (40 km, 50 MHz up, 300 MHz band)
  antennas, autos, timesteps, channels, pols, dtype ("c64" / "c128"), nan (fraction of non-finite samples)
  directions, spread (largest offset from the phase centre, radians)
  interval    timesteps per solution (0: one solution over all of them)
  host        visibilities in host memory; False: resident on the GPU
  fresh       the metadata (A, A1 and their pseudo-inverses) is built inside the call, as the command line
              does; False: built once and kept, as a program does that calibrates more than once
  batched, mixed, graph  the library's options; all False are its defaults (the reference's schedule)
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "icrar-leap-accelerate_amd"))

import leap_amd as la  # noqa: E402
import leap_torch  # noqa: E402

C_LIGHT = 299792458.0
EARTH_ROTATION = 7.2921150e-5
LATITUDE = math.radians(-26.7033)
CENTRE = (0.5, math.radians(-27.0))
SOURCES = 4


def _case(name, **kw):
    c = dict(kind="calibrate", array="disk", antennas=128, autos=True, timesteps=14, channels=48, pols=4, dtype="c128",
             nan=0.0, directions=1, spread=0.02, interval=0, host=False, fresh=False, batched=False, mixed=False,
             graph=False)
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One direction of a dozen antennas, one integration: what a call costs by itself.
        _case("tiny_call", antennas=12, autos=False, timesteps=1, channels=8, dtype="c64"),
        # The drop-in call as the command line makes it: columns in host memory, metadata inside the call,
        # default options, a few directions, two minutes of a 128-antenna array.
        _case("drop_in_host", dtype="c64", directions=4, host=True, fresh=True),
        # Default options on resident data with the metadata kept: a program looping over direction lists.
        _case("mwa_plain", directions=16),
        # A solution for every integration (the reference's own slice tests do this): many small solves.
        _case("mwa_timesteps", dtype="c64", directions=16, interval=1, batched=True),
        # Many directions of the same array in one pass, FP64, a narrow band of 48 channels.
        _case("mwa_batched_64", directions=64, batched=True),
        # Default options on a 256-station array with the measurement set's own complex64 data.
        _case("core_plain_c64", array="spiral", antennas=256, timesteps=32, channels=384, dtype="c64", directions=4),
        # The same on complex128 data, where the visibilities' bytes weigh most.
        _case("core_plain_c128", array="spiral", antennas=256, timesteps=32, channels=384, directions=2),
        # The benchmark's headline: 256 directions in one pass over the 51.7 GB complex64 cube, mixed precision.
        _case("core_mixed_256", array="spiral", antennas=256, timesteps=128, channels=384, dtype="c64", directions=256,
              batched=True, mixed=True),
        # Batched FP64 on a 51.7 GB complex128 cube, wide field, captured once and replayed.
        _case("core_fp64_64_graph", array="spiral", antennas=256, timesteps=64, channels=384, directions=64, spread=0.1,
              batched=True, graph=True),
        # Three uneven measurement sets in one call, mixed precision (the sizes given are the largest set's).
        _case("uneven_sets", kind="sets", array="spiral", antennas=256, timesteps=64, channels=96, dtype="c64",
              directions=64, spread=0.1, batched=True, mixed=True),
        # Direction and array refinement: loss, then its gradients by backward().
        _case("residual_grad", kind="grad", array="spiral", antennas=128, autos=False, timesteps=64, channels=192,
              dtype="c64", directions=16),
        # Odd sizes throughout: 2 pols, 131 channels, intervals that do not fill the observation, missing samples.
        _case("ragged_survey", array="spiral", antennas=61, autos=False, timesteps=37, channels=131, pols=2, dtype="c64",
              nan=1e-3, directions=21, interval=12, batched=True),
    ]


def draw(rng):
    """One more case: any kind, sizes spread over their ranges, at most the largest listed case's cost."""
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["calibrate", "calibrate", "calibrate", "sets", "grad"])
    batched = kind == "sets" or (kind == "calibrate" and rng.random() < 0.6)
    mixed = batched and rng.random() < 0.4
    host = kind == "calibrate" and rng.random() < 0.25
    fresh = kind == "calibrate" and rng.random() < 0.3
    # A host cube crosses the bus and is made again for every pass of the measurement: up to 1 GB of it.
    most = 1e9 if host else 3e9 if kind == "grad" else 2.6e10
    directions = log_int(1, 256) if batched else log_int(1, 40) if kind == "grad" else log_int(1, 16)
    dtype = "c64" if mixed or rng.random() < 0.5 else "c128"
    pols = rng.choice([1, 2, 4, 4])
    timesteps, channels = log_int(1, 128), log_int(8, 500)
    if not batched and not host:
        most /= max(1, directions)
    per = timesteps * channels * pols * (8 if dtype == "c64" else 16)
    antennas = max(8, min(log_int(8, 256), int(math.sqrt(2 * most / per))))
    return _case(None, kind=kind, array=rng.choice(["disk", "spiral"]), antennas=antennas,
                 autos=kind != "grad" and rng.random() < 0.5, timesteps=timesteps, channels=channels, pols=pols,
                 dtype=dtype, nan=rng.choice([0.0, 0.0, 1e-3]), directions=directions, spread=rng.choice([0.02, 0.1]),
                 interval=rng.choice([0, 0, log_int(max(1, timesteps // 16), timesteps)]) if kind == "calibrate" else 0,
                 host=host, fresh=fresh, batched=batched, mixed=mixed,
                 graph=batched and not host and not fresh and rng.random() < 0.25)


# ---- inputs -----------------------------------------------------------------


def _dd(centre, direction):
    """The rotation from the phase centre's to a direction's uvw frame."""
    a, b, c = math.pi / 2 - centre[1], direction[0] - centre[0], direction[1] - math.pi / 2

    def rx(t):
        return np.array([[1, 0, 0], [0, np.cos(t), -np.sin(t)], [0, np.sin(t), np.cos(t)]])

    return rx(c) @ np.array([[np.cos(b), np.sin(b), 0], [-np.sin(b), np.cos(b), 0], [0, 0, 1]]) @ rx(a)


def _set_sizes(case):
    """The measurement sets of a case: (antennas, autos, timesteps, channels) each."""
    one = (case["antennas"], case["autos"], case["timesteps"], case["channels"])
    if case["kind"] != "sets":
        return [one]
    n, t, c = case["antennas"], case["timesteps"], case["channels"]
    return [one, (max(8, n // 2), True, max(1, t // 5), max(8, c // 2)),
            (max(8, n // 7), False, max(1, t // 2), min(500, 3 * c + 12))]


def _columns(case, size, rng):
    """The measurement set's host columns, and the ENU-to-UVW matrices of its timesteps."""
    n, autos, T, C = size
    if case["array"] == "spiral":
        arm, j = np.arange(n) % 3, np.arange(n) // 3
        r = 20.0 * (20000.0 / 20.0) ** (j / max(1, (n + 2) // 3 - 1))
        th = arm * (2 * np.pi / 3) + 1.2 * np.log(r / 20.0) + 0.05 * (rng.random(n) - 0.5)
        f0, df = 50e6, 300e6 / C
    else:
        r, th = 750.0 * np.sqrt(rng.random(n)), 2 * np.pi * rng.random(n)
        f0, df = 169.6e6, 40e3
    enu = np.stack([r * np.cos(th), r * np.sin(th), np.zeros(n)], axis=1)
    a1, a2 = np.triu_indices(n, 0 if autos else 1)
    a1, a2 = a1.astype(np.int32), a2.astype(np.int32)
    nbl = len(a1)
    hour = EARTH_ROTATION * (np.arange(T) + 0.5 - 0.5 * T)
    sd, cd, sl, cl = math.sin(CENTRE[1]), math.cos(CENTRE[1]), math.sin(LATITUDE), math.cos(LATITUDE)
    sh, ch, o = np.sin(hour), np.cos(hour), np.zeros(T)
    W = np.stack([sh, ch, o, -sd * ch, sd * sh, o + cd, cd * ch, -cd * sh, o + sd], axis=1).reshape(T, 3, 3)
    M = W @ np.array([[0, -sl, cl], [1, 0, 0], [0, cl, sl]])
    ant = np.einsum("tij,aj->tai", M, enu)
    uvw = (ant[:, a2] - ant[:, a1]).reshape(T * nbl, 3)
    flag = (rng.random(nbl) < 0.02) & (a1 != a2) & (np.arange(nbl) >= n)
    return {"num_stations": n, "total_antennas": n, "num_baselines": nbl, "num_rows": nbl * T, "num_channels": C,
            "num_pols": case["pols"], "freq_start_hz": f0, "freq_inc_hz": df, "phase_centre": CENTRE, "antenna1": a1,
            "antenna2": a2, "time": np.repeat(5.0203e9 + np.arange(T), nbl), "flag": flag.astype(np.uint8),
            "uvw": np.ascontiguousarray(uvw)}, M


def _visibilities(case, ms, rng, gen):
    """The DATA column on the GPU, [row][channel][pol]: sources under per-antenna phase screens, plus noise."""
    R, C, P, nbl = ms["num_rows"], ms["num_channels"], ms["num_pols"], ms["num_baselines"]
    screen = rng.uniform(-np.pi, np.pi, ms["num_stations"])
    offsets = rng.uniform(-0.05, 0.05, (SOURCES, 2))
    flux = rng.uniform(1.0, 10.0, SOURCES)
    dz = np.stack([_dd(CENTRE, (CENTRE[0] + x, CENTRE[1] + y))[2] - [0, 0, 1] for x, y in offsets])
    path = torch.from_numpy(ms["uvw"]).cuda() @ torch.from_numpy(dz.T.copy()).cuda()  # [row][source], metres
    gain = torch.from_numpy(screen[ms["antenna1"]] - screen[ms["antenna2"]]).cuda().float()
    gain = torch.polar(torch.ones_like(gain), gain)
    kappa = (ms["freq_start_hz"] + ms["freq_inc_hz"] * torch.arange(C, device="cuda", dtype=torch.float64)) / C_LIGHT
    pol = torch.tensor([1.0, 0.1 + 0.03j, 0.08 - 0.06j, 0.9], device="cuda", dtype=torch.complex64)[:P]
    kind = torch.complex64 if case["dtype"] == "c64" else torch.complex128
    vis = torch.empty((R, C, P), device="cuda", dtype=kind)
    step = max(1, (1 << 25) // C)
    for r in range(0, R, step):
        at = slice(r, min(R, r + step))
        model = 0
        for s in range(SOURCES):
            turns = path[at, s, None] * kappa
            turns = ((turns - torch.round(turns)) * (2 * math.pi)).float()
            model = model + torch.polar(torch.full_like(turns, flux[s]), turns)
        model = model * gain[torch.arange(at.start, at.stop, device="cuda") % nbl, None]
        noise = torch.randn(model.shape + (P,), device="cuda", dtype=torch.complex64, generator=gen)
        vis[at] = torch.add(model[..., None] * pol, noise, alpha=0.15).to(kind)
        if case["nan"]:
            lost = torch.rand(model.shape + (P,), device="cuda", generator=gen) < case["nan"]
            vis[at] = torch.where(lost, torch.full((), float("nan"), device="cuda", dtype=kind), vis[at])
    return vis


def _inputs(case, seed):
    """Per measurement set: columns, visibilities on the GPU, directions, ENU-to-UVW matrices, offsets, deltas."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    sets = []
    for size in _set_sizes(case):
        ms, M = _columns(case, size, rng)
        vis = _visibilities(case, ms, rng, gen)
        D = case["directions"]
        dirs = np.asarray(CENTRE) + rng.uniform(-case["spread"], case["spread"], (D, 2))
        sets.append((ms, vis, dirs, M, rng.normal(0, 1e-4, (D, 2)), rng.normal(0, 0.01, (size[0], 3))))
    torch.cuda.synchronize()
    return sets


# ---- the calls --------------------------------------------------------------


def prepare(case, seed):
    ctx = la.Context(0)
    opts = la.options(strategy=la.LEAP_STRATEGY_BATCHED if case["batched"] else la.LEAP_STRATEGY_PER_DIRECTION,
                      precision=la.LEAP_PRECISION_MIXED if case["mixed"] else la.LEAP_PRECISION_FP64,
                      graph=1 if case["graph"] else 0)
    state = {"case": case, "ctx": ctx, "opts": opts, "keep": [], "sets": []}
    for ms, vis, dirs, M, offsets, delta in _inputs(case, seed):
        if case["host"]:
            view = la.view_from_arrays(dict(ms, vis=vis.cpu().numpy()))
        else:
            uvw = torch.from_numpy(ms["uvw"]).cuda()
            torch.cuda.synchronize()
            view = la.view_from_arrays(ms, vis_device=vis.data_ptr(), uvw_device=uvw.data_ptr(),
                                       vis_dtype=la.LEAP_VIS_C64 if case["dtype"] == "c64" else la.LEAP_VIS_C128)
            state["keep"] += [vis, uvw]
        md = None if case["fresh"] else ctx.metadata(view)
        state["sets"].append((md, view, dirs, (0, case["interval"] or -1, -1)))
        if case["kind"] == "grad":
            state["problem"] = leap_torch.CalibrationProblem(md=md, view=view, directions=dirs, enu_to_uvw=M)
            state["offsets"] = torch.from_numpy(offsets).requires_grad_()
            state["delta"] = torch.from_numpy(delta).requires_grad_()
    return state


def run(state):
    if state["case"]["kind"] == "grad":
        state["offsets"].grad = state["delta"].grad = None
        loss = leap_torch.residual_loss(state["offsets"], state["delta"], state["problem"])
        loss.backward()
        return loss.detach(), state["offsets"].grad, state["delta"].grad
    if state["case"]["kind"] == "sets":
        return state["ctx"].calibrate_batch(state["sets"], state["opts"])
    md, view, dirs, slice_ = state["sets"][0]
    return state["ctx"].calibrate(view, dirs, slice_, opts=state["opts"], md=md)


def work(case):
    """The cube, uvw and results once; per row and direction the cheaper of a direct sum over the channels and
    an FFT of twice the channels with 16 points a direction; the solve as a product with the pseudo-inverse."""
    size = 8 if case["dtype"] == "c64" else 16
    nbytes = flops = 0
    for n, autos, T, C in _set_sizes(case):
        nbl, D, P = n * (n + 1) // 2 if autos else n * (n - 1) // 2, case["directions"], case["pols"]
        solutions = max(1, T // (case["interval"] or T))
        rows = nbl * (solutions * case["interval"] if case["interval"] else T)
        fft = 2 ** math.ceil(math.log2(2 * C))
        sums = rows * min(8 * C * D, 5 * fft * math.log2(fft) + 200 * D)
        nbytes += rows * (C * P * size + 24) + solutions * D * n * 8
        flops += (2 if case["kind"] == "grad" else 1) * (sums + solutions * D * 2 * nbl * n)
    return {"bytes": nbytes, "flops": flops}


# ---- the same in 64 bits, plainly -------------------------------------------


def _solver(ms, ref_ant=None):
    """(A as pairs of antennas, the baselines of its rows, the pseudo-inverse's product) of the phase matrix."""
    a1, a2, n = ms["antenna1"].astype(np.int64), ms["antenna2"].astype(np.int64), ms["num_stations"]
    keep = (a1 != a2) & (ms["flag"] == 0)
    if ref_ant is not None:
        keep &= (a1 == ref_ant) | (a2 == ref_ant)
    rows = np.nonzero(keep)[0]
    i, j = torch.from_numpy(a1[rows]).cuda(), torch.from_numpy(a2[rows]).cuda()
    G = np.zeros((n, n))
    np.add.at(G, (a1[rows], a1[rows]), 1)
    np.add.at(G, (a2[rows], a2[rows]), 1)
    np.add.at(G, (a1[rows], a2[rows]), -1)
    np.add.at(G, (a2[rows], a1[rows]), -1)
    G[0 if ref_ant is None else ref_ant, 0 if ref_ant is None else ref_ant] += 1
    Gi = torch.from_numpy(np.linalg.pinv(G, hermitian=True)).cuda()

    def solve(y):  # [direction][row] -> [direction][antenna]; the constraint's value is 0
        b = torch.zeros((len(y), n), dtype=torch.float64, device="cuda")
        b.index_add_(1, i, y).index_add_(1, j, -y)
        return b @ Gi

    return i, j, torch.from_numpy(rows).cuda(), solve


def _z_offsets(dirs):
    """The third rows of the directions' rotations less the phase centre's, on the GPU: path = uvw . row."""
    return torch.from_numpy(np.stack([_dd(CENTRE, d)[2] - [0, 0, 1] for d in dirs])).cuda()


def _averages(ms, vis, uvw, dz, rows, grad=None):
    """Sum over the rows' channels of pol 0 rotated to every direction, [direction][baseline]; a sample with a
    NaN in any pol is left out.  Channels in blocks of 16: exp(i sf kappa) as a product of two exponentials.
    With grad, the loss's gradient by these sums: its gradients by uvw and by dz instead."""
    C, nbl, D = ms["num_channels"], ms["num_baselines"], len(dz)
    J = -(-C // 16)
    k0, dk = ms["freq_start_hz"] / C_LIGHT, ms["freq_inc_hz"] / C_LIGHT
    inner = torch.arange(16, device="cuda", dtype=torch.float64)[None, :, None] * dk
    outer = k0 + torch.arange(J, device="cuda", dtype=torch.float64)[None, :, None] * (16 * dk)
    out = torch.zeros((nbl, D), dtype=torch.complex128, device="cuda")
    by_uvw, by_dz = torch.zeros_like(uvw), torch.zeros_like(dz)
    step = max(1, (1 << 28) // (16 * D * (2 * J + 32)))
    for r in range(rows.start, rows.stop, step):
        e = min(rows.stop, r + step)
        at = torch.arange(r, e, device="cuda") % nbl
        v = vis[r:e].to(torch.complex128)
        v = torch.where(torch.isnan(v.real + v.imag).any(dim=2), 0, v[:, :, 0])
        v = torch.nn.functional.pad(v, (0, 16 * J - C)).reshape(e - r, J, 16)
        path = (uvw[r:e] @ dz.T).requires_grad_(grad is not None)
        sf = (-2 * math.pi * path)[:, None, :]
        z, y = sf * inner, sf * outer
        s = torch.matmul(v, torch.polar(torch.ones_like(z), z))
        s = (s * torch.polar(torch.ones_like(y), y)).sum(dim=1)
        if grad is None:
            out.index_add_(0, at, s)
        else:
            s.backward(grad.T[at])
            by_uvw[r:e] = path.grad @ dz
            by_dz += path.grad.T @ uvw[r:e]
    return out.T.contiguous() if grad is None else (by_uvw, by_dz)


def _solution(avg, solvers):
    """One interval's calibrations [direction][antenna] from its averages."""
    (i, j, rows, solve), (_, _, rows1, solve1) = solvers
    cal1 = solve1(torch.angle(avg[:, rows1]))
    turn = 2 * math.pi * (cal1[:, i] - cal1[:, j])
    # the reference takes row n of the averages, not row I(n), for the n-th equation
    return solve(torch.angle(torch.polar(torch.ones_like(turn), -turn) * avg[:, : len(rows)])) + cal1


def _calibrate(case, ms, vis, dirs):
    nbl, T = ms["num_baselines"], ms["num_rows"] // ms["num_baselines"]
    uvw, dz = torch.from_numpy(ms["uvw"]).cuda(), _z_offsets(dirs)
    solvers = _solver(ms), _solver(ms, ms["num_stations"] - 1)
    step = case["interval"] or T
    cals, epochs = [], []
    for s in range(T // step):
        cals.append(_solution(_averages(ms, vis, uvw, dz, range(s * step * nbl, (s + 1) * step * nbl)), solvers))
        epochs.append((ms["time"][s * step * nbl], ms["time"][((s + 1) * step - 1) * nbl]))
    return torch.stack(cals).cpu().numpy(), np.array(epochs)


def _loss_grad(ms, vis, dirs, M, offsets, delta):
    """The sum of squares of what the calibration leaves of the phases, and its gradients."""
    nbl = ms["num_baselines"]
    a1, a2 = torch.from_numpy(ms["antenna1"]).cuda().long(), torch.from_numpy(ms["antenna2"]).cuda().long()
    turn = torch.from_numpy(M).cuda()
    shift = torch.from_numpy(delta).cuda()
    uvw = torch.from_numpy(ms["uvw"]).cuda() + torch.matmul(shift[a2] - shift[a1], turn.mT).reshape(-1, 3)
    where = dirs + offsets
    dz, rows = _z_offsets(where), range(ms["num_rows"])
    avg = _averages(ms, vis, uvw, dz, rows).requires_grad_()
    solvers = _solver(ms), _solver(ms, ms["num_stations"] - 1)
    i, j, at, _ = solvers[0]
    cal = _solution(avg, solvers)
    rest = cal[:, i] - cal[:, j] - torch.angle(avg[:, at])
    loss = ((rest - 2 * math.pi * torch.round(rest / (2 * math.pi))) ** 2).sum()
    loss.backward()
    by_uvw, by_dz = _averages(ms, vis, uvw, dz, rows, grad=avg.grad)
    by_enu = torch.matmul(by_uvw.reshape(len(M), nbl, 3), turn).sum(dim=0)
    by_delta = torch.zeros_like(shift).index_add_(0, a2, by_enu).index_add_(0, a1, -by_enu)
    h = 1e-30  # the rotation's derivative by a complex step
    step = np.array([[np.imag(_dd(CENTRE, d + h * 1j * k)[2]) / h for k in np.eye(2)] for d in where])
    by_offset = torch.einsum("dk,dik->di", by_dz, torch.from_numpy(step).cuda())
    return loss.detach().cpu(), by_offset.cpu(), by_delta.cpu()


def exact(case, seed):
    sets = _inputs(case, seed)
    if case["kind"] == "grad":
        return _loss_grad(*sets[0])
    got = [_calibrate(case, *s[:3]) for s in sets]
    return got if case["kind"] == "sets" else got[0]
