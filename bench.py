#!/usr/bin/env python3
"""Benchmark of the gfx950 LEAP calibrator on the 256-station workload.

Workload (synthetic, generated on the device): 256 stations in a 40 km
three-arm log spiral, 32,896 baselines including autocorrelations, 128
timesteps of 1 s, 384 channels from 50 MHz at 781.25 kHz, 4 polarisations,
2% of baselines flagged, five point sources under per-antenna phase screens
plus noise.  One solution interval covers all 128 timesteps.

Default (headline): value is the batched mixed-precision rate — a step
calibrates 256 directions in one pass over the complex64 cube (51.7 GB
resident in HBM) — and the plain FP64 per-direction rate (a step = one
direction over the complex128 cube, 103.5 GB) is measured beside it in the
same run.  The JSON line carries the roofline of the dominant kernel from
HIP events on the library's stream, and a CPU baseline: the oracle on a
bounded sample of the same workload (host cores).
"""
import argparse
import json
import os
import platform
import sys
import time

import numpy as np

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "icrar-leap-accelerate_amd"))

import leap_amd as la  # noqa: E402

METRIC = "directions calibrated/s (256 st,128 t,384 ch) batched-mixed vs plain FP64; HBM GB/s"
HBM_PEAK_GBS = 8000.0
VALU_FP64_PEAK_TFLOPS = 78.6
# NUFFT flops per row and direction besides the weights and taps: shift factor 7,
# grid coordinate and offset 7, s^2 1, phasor 43, complex product 6, accumulation 2.
NUFFT_DIR_FLOPS = 66


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def c1_config():
    return dict(n_antennas=256, layout=1, array_radius_m=20000.0, autocorrelations=1, n_timesteps=128,
                integration_s=1.0, n_channels=384, freq_start_hz=50e6, freq_inc_hz=781.25e3, n_pols=4,
                flag_fraction=0.02, seed=1)


def directions(centre, n, seed=7, spread=0.02):
    rng = np.random.default_rng(seed)
    return np.column_stack([centre[0] + rng.uniform(-spread, spread, n), centre[1] + rng.uniform(-spread, spread, n)])


def traffic_from_profile(name):
    """HBM bytes per launch of a rotate kernel measured with rocprofv3 PMC counters, if committed."""
    p = os.path.join(REPO, "profiles", name)
    if not os.path.exists(p):
        return None
    try:
        return json.load(open(p)).get("bytes_per_launch")
    except (OSError, ValueError):
        return None


def host_cpu():
    """CPU model and core counts of this host (for the CPU baseline's label)."""
    model = platform.processor() or platform.machine()
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        usable = len(os.sched_getaffinity(0))
    except AttributeError:
        usable = os.cpu_count()
    return {"model": model, "nproc": usable, "logical_cpus": os.cpu_count()}


def c0_config():
    """The 128-antenna MWA-like set: 1.5 km disk, 8256 baselines with autos, 14 timesteps of 2 s, 48 channels
    from 169.6 MHz at 40 kHz, 4 pols, complex128, 1% of baselines flagged."""
    return dict(n_antennas=128, layout=0, array_radius_m=750.0, autocorrelations=1, n_timesteps=14,
                integration_s=2.0, n_channels=48, freq_start_hz=169.6e6, freq_inc_hz=40e3, n_pols=4,
                flag_fraction=0.01, seed=20201)


def run_c0(args):
    """The 128-antenna set in full: the oracle (1 thread) and the GPU (plain FP64 per direction, batched FP64),
    1 and 64 directions, the cube resident in host memory for the oracle and in HBM for the GPU."""
    sys.path.insert(0, os.path.join(REPO, "tests"))
    from oracle_bindings import Oracle  # the checker, used only for this reported baseline

    synth = la.SynthMS(**c0_config())
    synth.fill_host()
    ms = synth.host_dict()
    centre = ms["phase_centre"]
    o = Oracle()
    t = time.perf_counter()
    omd = o.metadata(ms)
    t_md = time.perf_counter() - t
    out = {"workload": "128 antennas / 8256 baselines (autos) / 14 t / 48 ch / 4 pol, complex128 (355 MB), "
                       "1 solution interval",
           "cpu": {"kind": "port", "threads": 1, "host": host_cpu(), "metadata_s": round(t_md, 3)}, "gpu": {}}
    for D in (1, 64):
        dirs = directions(centre, D, seed=55)
        t = time.perf_counter()
        for d in dirs:  # the Calibrate loop (CpuLeapCalibrator.cc:132-139) over prebuilt metadata
            omd.apply_inversion(omd.rotate(d))
        dt = time.perf_counter() - t
        out["cpu"][f"directions_per_s_{D}"] = round(D / dt, 3)
        log(f"[c0] oracle {D} direction(s): {dt:.2f} s after metadata")
    ctx = la.Context(0)
    vis_ptr = ctx.malloc(synth.num_rows * synth.num_channels * synth.num_pols * 16)
    uvw_ptr = ctx.malloc(synth.num_rows * 24)
    ctx.synth_fill_device(synth, la.LEAP_VIS_C128, vis_ptr, uvw_ptr)
    view = la.view_from_arrays(synth.host_dict(), vis_device=vis_ptr, vis_dtype=la.LEAP_VIS_C128, uvw_device=uvw_ptr)
    md = ctx.metadata(view)
    for name, D, opts in (("plain_fp64", 1, la.options()),
                          ("plain_fp64", 64, la.options()),
                          ("batched_fp64", 64, la.options(strategy=la.LEAP_STRATEGY_BATCHED))):
        dirs = directions(centre, D, seed=56)
        for _ in range(2):
            ctx.calibrate(view, dirs, md=md, opts=opts)
        reps = 10
        t = time.perf_counter()
        for _ in range(reps):
            ctx.calibrate(view, dirs, md=md, opts=opts)
        dt = (time.perf_counter() - t) / reps
        out["gpu"][f"{name}_directions_per_s_{D}"] = round(D / dt, 1)
    ctx.free(vis_ptr)
    ctx.free(uvw_ptr)
    ctx.close()
    return out


# The uneven batch of three sets: antennas, autocorrelations, timesteps, channels.
UNEVEN = [(36, 0, 32, 300), (128, 1, 14, 48), (256, 1, 64, 96)]


def run_c2(args):
    """Batching in FP64 and the uneven batch: 64 directions (offsets up to 0.1 rad) on the 256-station
    complex128 cube captured as one HIP graph and replayed each step; then the three uneven sets in one
    call per step, in FP64 (captured) on their complex128 cubes and in mixed precision on their complex64
    cubes (the automatic route: the NUFFT, width 16 in FP64, for the 300- and 96-channel sets, Horner for
    the 48-channel one)."""
    steps = args.steps
    out = {}
    synth = la.SynthMS(**c1_config())
    R, C, P = synth.num_rows, synth.num_channels, synth.num_pols
    ctx = la.Context(0)
    vis_ptr = ctx.malloc(R * C * P * 16)
    uvw_ptr = ctx.malloc(R * 24)
    ctx.synth_fill_device(synth, la.LEAP_VIS_C128, vis_ptr, uvw_ptr)
    view = la.view_from_arrays(synth.host_dict(), vis_device=vis_ptr, vis_dtype=la.LEAP_VIS_C128, uvw_device=uvw_ptr)
    md = ctx.metadata(view)
    dirs = directions((view.phase_centre_ra_rad, view.phase_centre_dec_rad), 64, seed=13, spread=0.1)
    opts = la.options(strategy=la.LEAP_STRATEGY_BATCHED, graph=1)
    for _ in range(max(1, args.warmup)):
        ctx.calibrate(view, dirs, md=md, opts=opts)
    step_s = []
    for _ in range(steps):
        t = time.perf_counter()
        ctx.calibrate(view, dirs, md=md, opts=opts)
        step_s.append(time.perf_counter() - t)
    replayed = ctx.last_graph() == 2
    route = ctx.last_route()[0]
    out["single_set"] = {"workload": "256 stations / 32896 baselines / 128 t / 384 ch / 4 pol, complex128 cube "
                                     "103.5 GB in HBM, 64 directions per step, FP64, one HIP graph replayed",
                         "graph_replayed": replayed, "tile": ctx.last_direction_block(),
                         "channel_sums": {la.LEAP_CHANNEL_SUM_NUFFT_W16: "width-16 NUFFT (FP64 transform)",
                                          la.LEAP_CHANNEL_SUM_HORNER: "FP64 Horner"}.get(route, str(route)),
                         "ms_per_step_median": round(float(np.median(step_s)) * 1e3, 3),
                         "directions_per_s": round(64 * steps / sum(step_s), 1)}
    log(f"[c2] 64 FP64 directions, graph: {out['single_set']['ms_per_step_median']} ms per step")
    ctx.free(vis_ptr)
    ctx.free(uvw_ptr)
    # the uneven batch, complex128 for FP64 and complex64 for mixed precision
    ptrs = []
    for name, prec, vd, elem in (("fp64", 0, la.LEAP_VIS_C128, 16), ("mixed", 1, la.LEAP_VIS_C64, 8)):
        batch = []
        for i, (n_ant, autos, T, Cs) in enumerate(UNEVEN):
            s = la.SynthMS(n_antennas=n_ant, autocorrelations=autos, n_timesteps=T, n_channels=Cs,
                           freq_start_hz=50e6, freq_inc_hz=781.25e3 * 384 / Cs, seed=60 + i)
            vp = ctx.malloc(s.num_rows * s.num_channels * s.num_pols * elem)
            up = ctx.malloc(s.num_rows * 24)
            ptrs += [vp, up]
            ctx.synth_fill_device(s, vd, vp, up)
            v = la.view_from_arrays(s.host_dict(), vis_device=vp, vis_dtype=vd, uvw_device=up)
            batch.append((ctx.metadata(v), v, directions((v.phase_centre_ra_rad, v.phase_centre_dec_rad), 64,
                                                          seed=70 + i, spread=0.1), (0, -1, -1)))
        bopts = la.options(precision=prec, strategy=la.LEAP_STRATEGY_BATCHED, graph=1 if prec == 0 else 0)
        for _ in range(max(1, args.warmup)):
            ctx.calibrate_batch(batch, bopts)
        step_s, k_ms = [], []
        for _ in range(steps):
            t = time.perf_counter()
            ctx.calibrate_batch(batch, bopts)
            step_s.append(time.perf_counter() - t)
            k_ms.append(ctx.last_kernel_times()[0])
        route = ctx.last_route()[0]
        out[f"uneven_batch_{name}"] = {
            "workload": "36 antennas / 630 baselines / 300 ch / 32 t; 128 / 8256 / 48 / 14; 256 / 32896 / 96 / 64; "
                        f"64 directions each, {'complex128' if elem == 16 else 'complex64'} cubes in HBM, one call "
                        "per step" + (" captured as a HIP graph" if prec == 0 else ""),
            "ms_per_step_median": round(float(np.median(step_s)) * 1e3, 3),
            "rotate_kernel_ms": None if prec == 0 else round(float(np.median(k_ms)), 4),
            "directions_per_s": round(3 * 64 * steps / sum(step_s), 1),
            "channel_sums": {la.LEAP_CHANNEL_SUM_NUFFT: "NUFFT (300- and 96-channel sets) + Horner (48 channels)",
                             la.LEAP_CHANNEL_SUM_NUFFT_W16: "width-16 NUFFT (300- and 96-channel sets) + FP64 Horner "
                                                            "(48 channels)"}.get(route, "FP64 Horner")}
        log(f"[c2] uneven batch {name}: {out[f'uneven_batch_{name}']['ms_per_step_median']} ms per step")
        for p_ in ptrs:
            ctx.free(p_)
        ptrs = []
    ctx.close()
    return out


def cpu_baseline(ctx, synth, vis_ptr, vis_dtype, timesteps):
    """The oracle (single thread) on the first `timesteps` timesteps of the same cube, scaled in T."""
    sys.path.insert(0, os.path.join(REPO, "tests"))
    from oracle_bindings import Oracle  # the checker, used only for this reported baseline

    nbl = synth.num_baselines
    rows = nbl * timesteps
    host = np.zeros((rows, synth.num_channels, synth.num_pols),
                    dtype=np.complex64 if vis_dtype == la.LEAP_VIS_C64 else np.complex128)
    ctx.d2h(host, vis_ptr)
    ms = dict(synth.host_dict(host))
    ms["num_rows"] = rows
    ms["uvw"] = synth.uvw[:rows]
    ms["time"] = synth.time[:rows]
    o = Oracle()
    t = time.perf_counter()
    md = o.metadata(ms)
    t_md = time.perf_counter() - t
    d = directions(ms["phase_centre"], 1, seed=99)[0]
    t = time.perf_counter()
    avg = md.rotate(d)
    t_rot = time.perf_counter() - t
    t = time.perf_counter()
    md.apply_inversion(avg)
    t_inv = time.perf_counter() - t
    T = synth.cfg.n_timesteps
    per_dir = t_rot * (T / timesteps) + t_inv
    return {
        "value": 1.0 / per_dir,
        "unit": "directions/s",
        "cores": 1,
        "kind": "port",
        "host": host_cpu(),
        "sample": (f"oracle (FP64 C++ restatement, 1 thread of {host_cpu()['model']}) on "
                   f"{timesteps} of {T} timesteps of the same cube, 1 direction; RotateVisibilities time "
                   f"{t_rot:.2f} s scaled x{T // timesteps} in T plus inversion {t_inv * 1e3:.1f} ms; "
                   f"one-off metadata (SVD pseudo-inverse) {t_md:.1f} s not counted"),
    }


def copy_probe(gb):
    """hipMemcpy device-to-device of a known size, 3 times; prints the byte count and the best
    read + write rate (host clock around each synchronous copy)."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so")
    n = int(gb * 1e9) // 4096 * 4096
    ctx = la.Context(0)
    a = ctx.malloc(n)
    b = ctx.malloc(n)
    best = None
    for _ in range(3):
        t = time.perf_counter()
        rc = hip.hipMemcpy(ctypes.c_void_p(b), ctypes.c_void_p(a), ctypes.c_size_t(n), 3)  # device to device
        hip.hipDeviceSynchronize()
        dt = time.perf_counter() - t
        if rc != 0:
            raise RuntimeError(f"hipMemcpy failed: {rc}")
        best = dt if best is None else min(best, dt)
    ctx.free(a)
    ctx.free(b)
    print(json.dumps({"copy_probe_bytes": n, "copies": 3, "best_read_write_gbs": round(2 * n / best / 1e9, 1)}),
          flush=True)
    return 0


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20, help="timed steps of each leg")
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--mode", default="headline",
                    choices=["headline", "plain", "batched-fp64", "batched-mixed", "adjoint"],
                    help="headline: batched-mixed (value) measured beside plain; plain: FP64 per direction on "
                         "the complex128 cube; batched-fp64: FP64, one pass per block of directions on the "
                         "complex128 cube; batched-mixed: mixed precision on the complex64 cube; adjoint: "
                         "calibration-residual loss and its gradients (128 stations, 16 directions)")
    ap.add_argument("--directions", type=int, default=0, help="directions per step (default 1 plain, 64 "
                    "batched-fp64, 256 batched-mixed)")
    ap.add_argument("--direction-block", type=int, default=0, help="0 = autotuned")
    ap.add_argument("--lane-directions", type=int, default=0, help="directions per lane (0 = autotuned)")
    ap.add_argument("--fp32-blocks", action="store_true",
                    help="batched-mixed only: FP32 Horner blocks re-anchored every 32 channels instead of the "
                         "full-row FP64 Horner")
    ap.add_argument("--direct-cube", action="store_true",
                    help="batched: run the Horner kernel straight from the cube (no pol-0 pack)")
    ap.add_argument("--pack-timesteps", type=int, default=0, help="timesteps per pack chunk (0 = automatic)")
    ap.add_argument("--channel-sum", default="auto", choices=["auto", "horner", "nufft", "nufft-fp32", "nufft-w16"],
                    help="mixed precision: channel sums by FP64 Horner or the NUFFT (auto: NUFFT where supported)")
    ap.add_argument("--host-cube", action="store_true",
                    help="batched modes: the cube stays in (pageable) host memory and every step stages it "
                         "(PCIe-inclusive rate; not the headline value, which has the cube resident in HBM)")
    ap.add_argument("--no-error-check", dest="error_check", action="store_false",
                    help="batched-mixed: skip the per-direction error against the plain FP64 path")
    ap.add_argument("--no-c0", dest="c0", action="store_false",
                    help="headline: skip the 128-antenna set timed in full on the oracle and the GPU")
    ap.add_argument("--no-c2", dest="c2", action="store_false",
                    help="headline: skip 64 FP64 directions under graph capture and the uneven three-set batch")
    ap.add_argument("--cpu-timesteps", type=int, default=2, help="timesteps in the CPU-baseline sample (0 = skip)")
    ap.add_argument("--copy-probe-gb", type=float, default=0.0,
                    help="only run device-to-device copies of this size (calibrates rocprofv3 FETCH_SIZE / "
                         "WRITE_SIZE against a copy of known bytes) and exit")
    args = ap.parse_args()
    if args.copy_probe_gb > 0:
        return copy_probe(args.copy_probe_gb)
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported in this build "
              "(the per-GPU work is the same for every GPU count: directions or rows shard without "
              "changing a GPU's kernel).", file=sys.stderr)
        return 2

    if args.mode == "adjoint":
        print(json.dumps(run_adjoint(args)), flush=True)
        return 0
    if args.mode == "headline":
        plain = run_mode(args, "plain", 1, with_cpu=False)
        mixed = run_mode(args, "batched-mixed", args.directions or 256, with_cpu=args.cpu_timesteps > 0)
        out = mixed
        out["config"]["plain_fp64"] = {
            "directions_per_s": plain["value"], "ms_per_step": plain["ms_per_step"],
            "rotate_kernel_ms": plain["roofline"]["kernel_ms"], "roofline": plain["roofline"],
        }
        out["config"]["speedup_vs_plain_fp64"] = round(mixed["value"] / plain["value"], 2)
        if args.c0:
            out["config"]["c0"] = run_c0(args)
        if args.c2:
            out["config"]["c2"] = run_c2(args)
        out["config"]["workload"] = ("batched mixed-precision calibration (complex64 cube 51.7 GB resident in "
                                     f"HBM, {out['config']['directions_per_step']} directions per step, one pass "
                                     "over the cube) vs plain FP64 per-direction calibration (complex128 cube "
                                     "103.5 GB, 1 direction per step); 256 stations / 32896 baselines (autos) / "
                                     "128 t / 384 ch / 4 pol, 1 solution interval")
    else:
        D = args.directions or {"plain": 1, "batched-fp64": 64, "batched-mixed": 256}[args.mode]
        out = run_mode(args, args.mode, D, with_cpu=args.cpu_timesteps > 0)
    print(json.dumps(out), flush=True)
    return 0


def run_mode(args, mode, D, with_cpu, steps=None):
    steps = steps or args.steps
    vis_dtype = la.LEAP_VIS_C64 if mode == "batched-mixed" else la.LEAP_VIS_C128
    elem = 8 if vis_dtype == la.LEAP_VIS_C64 else 16
    opts = la.options(precision=la.LEAP_PRECISION_MIXED if mode == "batched-mixed" else la.LEAP_PRECISION_FP64,
                      strategy=la.LEAP_STRATEGY_PER_DIRECTION if mode == "plain" else la.LEAP_STRATEGY_BATCHED,
                      direction_block=args.direction_block)
    opts.fp32_blocks = 1 if args.fp32_blocks else 0
    opts.lane_directions = args.lane_directions
    opts.direct_cube = 1 if args.direct_cube else 0
    opts.pack_timesteps = args.pack_timesteps
    opts.channel_sum = {"auto": 0, "horner": 1, "nufft": 2, "nufft-fp32": 3, "nufft-w16": 4}[args.channel_sum]

    cfg = c1_config()
    log(f"[{mode}] building synthetic measurement set (host columns)")
    synth = la.SynthMS(**cfg)
    R, C, P, nbl = synth.num_rows, synth.num_channels, synth.num_pols, synth.num_baselines
    ctx = la.Context(0)
    vis_bytes = R * C * P * elem
    log(f"[{mode}] allocating {vis_bytes / 1e9:.1f} GB {'complex64' if elem == 8 else 'complex128'} cube on the "
        "device and generating it")
    vis_ptr = ctx.malloc(vis_bytes)
    uvw_ptr = ctx.malloc(R * 3 * 8)
    t = time.perf_counter()
    ctx.synth_fill_device(synth, vis_dtype, vis_ptr, uvw_ptr)
    log(f"[{mode}] cube generated in {time.perf_counter() - t:.2f} s")
    view = la.view_from_arrays(synth.host_dict(), vis_device=vis_ptr, vis_dtype=vis_dtype, uvw_device=uvw_ptr)
    host_vis = None
    if args.host_cube:
        host_vis = np.empty((R, C, P), dtype=np.complex64 if elem == 8 else np.complex128)
        t = time.perf_counter()
        ctx.d2h(host_vis, vis_ptr)
        log(f"[{mode}] cube copied to host memory in {time.perf_counter() - t:.2f} s")
        view = la.view_from_arrays(synth.host_dict(host_vis))
    t = time.perf_counter()
    md = ctx.metadata(view)
    t_md = time.perf_counter() - t
    log(f"[{mode}] metadata (A {md.K}x{md.N}, A1 {md.K1}x{md.N}, pseudo-inverses) in {t_md:.2f} s")

    dirs = directions((view.phase_centre_ra_rad, view.phase_centre_dec_rad), (args.warmup + steps) * D)
    for i in range(args.warmup):
        ctx.calibrate(view, dirs[i * D:(i + 1) * D], md=md, opts=opts)
        log(f"[{mode}] warmup step {i + 1}/{args.warmup} done")
    rot_ms, pack_ms, staged, step_s = [], [], [], []
    t0 = time.perf_counter()
    for i in range(steps):
        j = args.warmup + i
        ts = time.perf_counter()
        ctx.calibrate(view, dirs[j * D:(j + 1) * D], md=md, opts=opts)  # returns after a stream sync
        step_s.append(time.perf_counter() - ts)
        avg_ms, launches, _ = ctx.last_kernel_times()
        # device time of the rotate/average launches of one step (the plain path launches one per direction)
        rot_ms.append(avg_ms if mode == "plain" else avg_ms * launches)
        p_avg, p_n = ctx.last_pack_times()
        pack_ms.append(p_avg * p_n)
        staged.append(ctx.last_staged_bytes())
    elapsed = time.perf_counter() - t0
    log(f"[{mode}] {steps} timed steps of {D} directions in {elapsed:.3f} s")
    value = steps * D / elapsed
    k_ms = float(np.mean(rot_ms))
    tile = ctx.last_direction_block()
    route_cs, route_dc = ctx.last_route() if mode != "plain" else (0, 0)
    nufft = mode != "plain" and route_cs in (la.LEAP_CHANNEL_SUM_NUFFT, la.LEAP_CHANNEL_SUM_NUFFT_FP32,
                                             la.LEAP_CHANNEL_SUM_NUFFT_W16)
    nufft32 = nufft and route_cs == la.LEAP_CHANNEL_SUM_NUFFT_FP32
    nufft16 = nufft and route_cs == la.LEAP_CHANNEL_SUM_NUFFT_W16
    packed = (mode != "plain" and not args.fp32_blocks and not route_dc and tile in (641, 1282, 2564))
    if nufft:
        # NUFFT channel sums: per row one N-point complex FFT (5 N log2 N flops,
        # the conventional count) and per row and direction the weight
        # polynomials (W^2 / 2 FMAs), the W-tap interpolation (2 W FMAs) and
        # NUFFT_DIR_FLOPS of shift factor, grid coordinate, phasor and
        # accumulation (FMA = 2 flops).  The roofline's bound is HBM: the
        # algorithmic bytes (the cube once, uvw, pol 0 of avgData) over the
        # kernel time against 8 TB/s; the vector-ALU rate is reported beside it.
        plan = la.nufft_plan(C, fp32=nufft32, w16=nufft16)
        n_grid, width = plan["N"], plan["W"]
        per_row = 5 * n_grid * np.log2(n_grid)
        per_dir = 2 * (width * width // 2 + 2 * width) + NUFFT_DIR_FLOPS
        alg_flops = int(R * (per_row + D * per_dir))
        tflops = alg_flops / (k_ms * 1e-3) / 1e12
        src_bytes = R * C * P * elem if route_dc else R * C * 16
        # calibrations on this route keep pol 0 of avgData only (16 B per direction and baseline)
        alg_bytes = src_bytes + R * 24 + D * nbl * 16
        gbs = alg_bytes / (k_ms * 1e-3) / 1e9
        kname = ("rotate_average_nufft<float>" if nufft32 else
                 "rotate_average_nufft<double>, width 16" if nufft16 else "rotate_average_nufft<double>")
        prof = ("rotate_average_nufft32_c1" if nufft32 else
                "rotate_average_nufft_w16_c2" if nufft16 else "rotate_average_nufft_c1")
        roofline = {"kernel": kname, "bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS,
                    "unit": "GB/s", "frac": round(gbs / HBM_PEAK_GBS, 4),
                    "traffic": traffic_from_profile(prof + "_traffic.json"),
                    "kernel_ms": round(k_ms, 4), "algorithmic_bytes_per_launch": alg_bytes,
                    # measured with rocprofv3 counters, not live
                    "limiter": f"{'HBM' if nufft16 else 'vector ALU and LDS'} (profiles/{prof}.md)",
                    "valu": {"achieved_tflops": round(tflops, 2), "peak_tflops": VALU_FP64_PEAK_TFLOPS,
                             "frac": round(tflops / VALU_FP64_PEAK_TFLOPS, 4),
                             "algorithmic_flops_per_launch": alg_flops},
                    "nufft": {"transform": "fp32" if nufft32 else "fp64", "grid": n_grid, "width": width,
                              "fft_flops_per_row": int(per_row), "flops_per_row_direction": per_dir,
                              "source": (("complex64" if elem == 8 else "complex128") + " cube") if route_dc
                              else "packed pol-0 rows"},
                    # the direct sum's 8 flops per (row, channel, direction) over the kernel time
                    "direct_sum_equivalent_tflops": round(8 * R * C * D / (k_ms * 1e-3) / 1e12, 1)}
    elif mode == "plain":
        alg_bytes = R * C * P * elem + R * 24 + D * nbl * P * 16 + C * 8
        achieved = alg_bytes / (k_ms * 1e-3) / 1e9
        roofline = {"kernel": "rotate_average_f64", "bound": "hbm", "achieved": round(achieved, 1),
                    "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                    "traffic": traffic_from_profile("rotate_average_f64_c1_traffic.json"),
                    "kernel_ms": round(k_ms, 4), "algorithmic_bytes_per_launch": alg_bytes}
    else:
        # One complex multiply-accumulate (8 flops) per visibility, direction and pass.
        alg_flops = 8 * R * C * D
        achieved = alg_flops / (k_ms * 1e-3) / 1e12
        alg_bytes = R * C * P * elem + R * 24 + D * nbl * P * 16
        if packed:
            kernel, prof = "rotate_average_packed", "rotate_average_packed_c1_traffic.json"
            # the Horner kernel reads the packed pol-0 array (16 B per row and channel) instead of the cube
            alg_bytes = R * C * 16 + R * 24 + D * nbl * P * 16
        elif args.fp32_blocks:
            kernel, prof = "rotate_average_batched", None
        else:
            # counters of the complex64 (256 directions) and complex128 (64 directions) cubes
            kernel = "rotate_average_horner64"
            prof = "rotate_average_horner64_c2_traffic.json" if elem == 16 else "rotate_average_horner64_c1_traffic.json"
        roofline = {"kernel": kernel,
                    "bound": "valu-fp64", "achieved": round(achieved, 2), "peak": VALU_FP64_PEAK_TFLOPS,
                    "unit": "TFLOP/s", "frac": round(achieved / VALU_FP64_PEAK_TFLOPS, 4),
                    "traffic": traffic_from_profile(prof) if prof else None,
                    "kernel_ms": round(k_ms, 4), "algorithmic_flops_per_launch": alg_flops,
                    "hbm_gbs": round(alg_bytes / (k_ms * 1e-3) / 1e9, 1)}
    if packed and mode != "plain":
        p_ms = float(np.mean(pack_ms))
        pack_bytes = R * C * (P * elem + 16)  # read every pol once, write pol 0 as FP64 complex
        roofline["pack"] = {"kernel": "pack_pol0_kernel", "bound": "hbm", "ms": round(p_ms, 4),
                            "algorithmic_bytes": pack_bytes,
                            "achieved": round(pack_bytes / (p_ms * 1e-3) / 1e9, 1) if p_ms > 0 else None,
                            "peak": HBM_PEAK_GBS, "unit": "GB/s",
                            "frac": round(pack_bytes / (p_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4) if p_ms > 0 else None}

    error = None
    fp64_batched = None
    if mode == "batched-mixed" and args.error_check:
        # Outside the timed region: the first timed step's directions again, against the plain FP64 path
        # (the reference's arithmetic, held to 1e-9 rad of the oracle by the parity tests) on the same cube.
        j = args.warmup
        sel = dirs[j * D:(j + 1) * D]
        got, _ = ctx.calibrate(view, sel, md=md, opts=opts)
        t = time.perf_counter()
        want, _ = ctx.calibrate(view, sel, md=md, opts=la.options())
        log(f"[{mode}] FP64 reference of {D} directions in {time.perf_counter() - t:.2f} s")
        err = np.abs((got[0] - want[0] + np.pi) % (2 * np.pi) - np.pi)  # [D][N]
        per_max = err.max(axis=1)
        per_rms = np.sqrt((err ** 2).mean(axis=1))
        error = {"against": "plain FP64 GPU path on the same complex64 cube (1e-9 rad of the FP64 oracle in the "
                            "parity tests)",
                 "directions": D, "max_rad": float(per_max.max()), "rms_rad": float(np.sqrt((err ** 2).mean())),
                 "per_direction_max_rad": [float(f"{x:.3g}") for x in per_max],
                 "per_direction_rms_rad": [float(f"{x:.3g}") for x in per_rms]}
        log(f"[{mode}] wrapped phase error vs FP64: max {error['max_rad']:.3e} rad, rms {error['rms_rad']:.3e} rad")
        # FP64 precision on the same cube and directions, batched (its automatic route), also outside the
        # timed region: its rate beside the headline's, and its distance from the plain FP64 path.
        f64_opts = la.options(strategy=la.LEAP_STRATEGY_BATCHED)
        ctx.calibrate(view, sel, md=md, opts=f64_opts)  # tunes its tile
        f64_s = []
        for _ in range(5):
            t = time.perf_counter()
            f64, _ = ctx.calibrate(view, sel, md=md, opts=f64_opts)
            f64_s.append(time.perf_counter() - t)
        f64_err = np.abs((f64[0] - want[0] + np.pi) % (2 * np.pi) - np.pi)
        fp64_batched = {
            "workload": f"batched FP64 calibration of the same {D} directions on the same complex64 cube "
                        "(5 steps after a tuning call, not part of value)",
            "channel_sums": {la.LEAP_CHANNEL_SUM_NUFFT_W16: "width-16 NUFFT (FP64 transform)",
                             la.LEAP_CHANNEL_SUM_HORNER: "FP64 Horner"}.get(ctx.last_route()[0], "other"),
            "ms_per_step_median": round(float(np.median(f64_s)) * 1e3, 3),
            "directions_per_s": round(D / float(np.median(f64_s)), 1),
            "max_rad_vs_plain_fp64": float(f64_err.max())}
        log(f"[{mode}] batched FP64 on the same cube: {fp64_batched['ms_per_step_median']} ms per step, "
            f"max {fp64_batched['max_rad_vs_plain_fp64']:.2e} rad from the plain path")

    cpu = None
    if with_cpu:
        log(f"[{mode}] CPU baseline: oracle on {args.cpu_timesteps} timesteps")
        cpu = cpu_baseline(ctx, synth, vis_ptr, vis_dtype, args.cpu_timesteps)
        log(f"[{mode}] CPU baseline done")
    ctx.free(vis_ptr)
    ctx.free(uvw_ptr)
    ctx.close()

    host_note = None
    if args.host_cube:
        host_note = {"staged_bytes_per_step": int(np.mean(staged)),
                     "staged_gbs": round(float(np.mean(staged)) / (elapsed / steps) / 1e9, 1),
                     "note": "cube in pageable host memory, staged every step (pol 0 only on the packed path)"}
        del host_vis
    workload = {
        "plain": "plain FP64 per-direction calibration, complex128 cube 103.5 GB resident in HBM, 1 direction per step",
        "batched-fp64": f"batched FP64 calibration, complex128 cube 103.5 GB resident in HBM, {D} directions per "
                        "step in one pass over the cube",
        "batched-mixed": f"batched mixed-precision calibration, complex64 cube 51.7 GB resident in HBM, {D} "
                         "directions per step in one pass over the cube",
    }[mode]
    if args.host_cube:
        workload = workload.replace("resident in HBM", "in host memory, staged to the device every step")
    return {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "directions/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": args.warmup,
        "ms_per_step": round(elapsed / steps * 1e3, 3),
        "step_ms": {"median": round(float(np.median(step_s)) * 1e3, 3), "min": round(min(step_s) * 1e3, 3),
                    "max": round(max(step_s) * 1e3, 3), "mean": round(float(np.mean(step_s)) * 1e3, 3)},
        "value_median": round(D / float(np.median(step_s)), 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if mode != "batched-mixed" else (("c64 storage, f64 phase, f32 NUFFT transform" if nufft32
                                                         else "c64 storage, f64 phase and NUFFT") if nufft else
                                                        "c64 storage, f64 phase and Horner"),
        "data": "synthetic (seeded point sources x per-antenna phase screens + noise, generated on the device)",
        "config": {
            "workload": workload + "; 256 stations / 32896 baselines (autos) / 128 t / 384 ch / 4 pol, "
                        "1 solution interval",
            "stations": 256, "baselines": nbl, "timesteps": 128, "channels": C, "pols": P, "rows": R,
            "vis_dtype": "complex64" if elem == 8 else "complex128", "directions_per_step": D, "mode": mode,
            "tile": tile, "metadata_s": round(t_md, 3),
            **({"error_vs_fp64": error} if error else {}),
            **({"fp64_batched_same_cube": fp64_batched} if fp64_batched else {}),
        },
        "roofline": roofline,
        "cpu_baseline": cpu,
        **({"host_cube": host_note} if host_note else {}),
    }


def run_adjoint(args):
    """Loss + gradient evaluations of leap_hip_residual_loss_grad: 128 stations without
    autocorrelations (8128 baselines), 64 timesteps of 2 s, 192 channels, complex64 cube generated
    on the device, 16 directions, direction offsets N(0, 1e-4 rad), antenna position corrections
    N(0, 0.01 m).  A step is one forward (rotate, average, inversion, loss) and backward (adjoint
    of the inversion, then of rotate/average) pass, in the library's automatic adjoint mode (here
    the forward pass keeps each row's channel sums and the adjoint reads them); the same steps with
    the adjoint recomputing the phasors from the cube are timed beside it (config.recompute)."""
    cfg = dict(n_antennas=128, autocorrelations=0, n_timesteps=64, n_channels=192, seed=4)
    D = args.directions or 16
    synth = la.SynthMS(**cfg)
    nbl, R, C, P = synth.num_baselines, synth.num_rows, synth.num_channels, synth.num_pols
    ctx = la.Context(0)
    vis_ptr = ctx.malloc(R * C * P * 8)
    uvw_ptr = ctx.malloc(R * 3 * 8)
    ctx.synth_fill_device(synth, la.LEAP_VIS_C64, vis_ptr, uvw_ptr)
    view = la.view_from_arrays(synth.host_dict(), vis_device=vis_ptr, vis_dtype=la.LEAP_VIS_C64, uvw_device=uvw_ptr)
    rng = np.random.default_rng(4)
    centre = (view.phase_centre_ra_rad, view.phase_centre_dec_rad)
    dirs = directions(centre, D, seed=4)
    off = rng.normal(0, 1e-4, (D, 2))
    md = ctx.metadata(view)
    dp = rng.normal(0, 0.01, (md.N, 3))
    M = synth.enu_to_uvw
    for i in range(args.warmup):
        md.loss_grad(view, dirs, M, off, dp)
        log(f"[adjoint] warmup step {i + 1}/{args.warmup} done")
    steps = args.steps
    fwd_k, adj_k = [], []
    t = time.perf_counter()
    for _ in range(steps):
        md.loss_grad(view, dirs, M, off, dp)  # returns host values: every step ends synchronised
        f_ms, a_ms = ctx.last_loss_grad_times()
        fwd_k.append(f_ms)
        adj_k.append(a_ms)
    elapsed = time.perf_counter() - t
    t = time.perf_counter()
    for _ in range(steps):
        md.loss_grad(view, dirs, M, off, dp, want_grad=False)
    fwd = time.perf_counter() - t
    ctx.set_adjoint_mode(la.LEAP_ADJOINT_RECOMPUTE)
    rf_k, ra_k = [], []
    t = time.perf_counter()
    for _ in range(steps):
        md.loss_grad(view, dirs, M, off, dp)
        f_ms, a_ms = ctx.last_loss_grad_times()
        rf_k.append(f_ms)
        ra_k.append(a_ms)
    rec = time.perf_counter() - t
    ctx.set_adjoint_mode(la.LEAP_ADJOINT_AUTO)
    log(f"[adjoint] {steps} timed steps in {elapsed:.3f} s (forward only {fwd:.3f} s, recomputing adjoint "
        f"{rec:.3f} s)")
    cpu = None
    if args.cpu_timesteps > 0:
        sys.path.insert(0, os.path.join(REPO, "tests"))
        from oracle_bindings import Oracle  # the checker, used only for this reported baseline

        ts = args.cpu_timesteps
        rows = nbl * ts
        host = np.zeros((rows, C, P), dtype=np.complex64)
        ctx.d2h(host, vis_ptr)
        ms = dict(synth.host_dict(host))
        ms["num_rows"] = rows
        ms["uvw"] = synth.uvw[:rows]
        ms["time"] = synth.time[:rows]
        t = time.perf_counter()
        Oracle().loss_grad(ms, dirs, M, off, dp)
        t_cpu = time.perf_counter() - t
        scale = cfg["n_timesteps"] / ts
        cpu = {"value": 1.0 / (t_cpu * scale), "unit": "evaluations/s", "cores": 1, "kind": "port",
               "sample": (f"oracle loss and explicit gradient (FP64 C++ restatement, 1 thread) on {ts} of "
                          f"{cfg['n_timesteps']} timesteps, {D} directions, metadata included: {t_cpu:.2f} s "
                          f"scaled x{scale:g} in T")}
    ctx.free(vis_ptr)
    ctx.free(uvw_ptr)
    ctx.close()
    # Roofline of the dominant kernel, the forward pass with row sums (HBM): it reads the cube and
    # uvw, writes avgData and each row's sums (e0 P, e0 z P', 32 bytes per row and direction); P and
    # P' by Horner's rule would be 16 flop per (row, channel, direction), reported against the FP64
    # vector peak.  The adjoint kernel reads the row sums, uvw and abar and writes
    # the uvw gradient and the per-baseline dz partials.  Kernel times from the device's clock.
    a_ms, f_ms = float(np.median(adj_k)), float(np.median(fwd_k))
    q_bytes = R * D * 32
    fwd_bytes = R * C * P * 8 + R * 24 + D * nbl * P * 16 + q_bytes
    fwd_flops = 16 * R * C * D
    adj_bytes = q_bytes + R * 24 + D * nbl * 16 + R * 24 + nbl * D * 24
    roofline = {"kernel": "horner_wave_kernel (row sums kept)", "bound": "hbm",
                "achieved": round(fwd_bytes / (f_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(fwd_bytes / (f_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4), "traffic": None,
                "kernel_ms": round(f_ms, 4), "algorithmic_bytes_per_launch": fwd_bytes,
                "valu": {"achieved_tflops": round(fwd_flops / (f_ms * 1e-3) / 1e12, 2), "peak_tflops": 78.6,
                         "frac": round(fwd_flops / (f_ms * 1e-3) / 1e12 / 78.6, 4),
                         "algorithmic_flops_per_launch": fwd_flops},
                "adjoint": {"kernel": "adjoint_q_kernel (from the row sums)", "kernel_ms": round(a_ms, 4),
                            "algorithmic_bytes_per_launch": adj_bytes,
                            "achieved": round(adj_bytes / (a_ms * 1e-3) / 1e9, 1),
                            "frac": round(adj_bytes / (a_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)}}
    return {
        "metric": "calibration-residual loss + gradient evaluations/s (128 st, 8128 bl, 64 t, 192 ch, 16 dirs)",
        "value": round(steps / elapsed, 3),
        "unit": "evaluations/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": args.warmup,
        "ms_per_step": round(elapsed / steps * 1e3, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64 storage, f64 arithmetic",
        "data": "synthetic (seeded point sources x per-antenna phase screens + noise, generated on the device)",
        "config": {"workload": f"loss and gradients w.r.t. {D} direction offsets and 128 x 3 antenna positions; "
                               "128 stations / 8128 baselines (no autos) / 64 t / 192 ch / 4 pol, complex64 cube "
                               "resident in HBM",
                   "stations": 128, "baselines": nbl, "timesteps": 64, "channels": C, "pols": P,
                   "directions": D, "forward_only_ms": round(fwd / steps * 1e3, 3),
                   "adjoint_mode": "automatic: row sums kept by the forward pass",
                   "recompute": {"ms_per_step": round(rec / steps * 1e3, 3),
                                 "forward_kernel_ms": round(float(np.median(rf_k)), 4),
                                 "adjoint_kernel_ms": round(float(np.median(ra_k)), 4),
                                 "note": "the adjoint reads the cube again and recomputes the phasors, P and P'"}},
        "roofline": roofline,
        "cpu_baseline": cpu,
    }


if __name__ == "__main__":
    sys.exit(main())
