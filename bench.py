#!/usr/bin/env python
"""Benchmark of the ATV continuous max-flow on one GPU.

Workload (one step): the grid search of the reference experiment on one
128^3 helix phantom (tube radius 6, helix radius 32, pitch 48, noise sigma
1.5): 25 nt_weightings x 17 nt_decays = 425 ATV solves (a = 10^-1.5) of 500
iterations each, run as one batched solve on device-resident inputs. The
shared inputs (frames from Frangi -> adjustment -> GVF -> completion,
capacities, |grad I|^2) are prepared once, outside the timed region.

Reported beside it: every cell's fast Dice against the noise-free mask
(counted on the device); the same solves run one at a time (device-resident,
and through the numpy drop-in API); the 64^3 and 256^3 single solves through
the whole pipeline (the plain workloads, 500 and 1000 iterations); a ragged
set of helix phantoms through the whole pipeline with one packed max-flow
solve; serving latency (p50/p99) and throughput under Poisson arrivals of
mixed-size cuts, and of requests that need the whole preparation; the HBM
roofline of the max-flow iteration (84 algorithmic bytes per voxel-iteration)
with the HBM traffic rocprofv3 measured for the same kernels; and the CPU
oracle timed on a bounded sample on this host.

``--only PART`` runs one part (grid, plain, plain64, plain256, ragged, serve,
cpu; sigmas: the ATV and the TV grid at all 15 noise levels of the experiment,
not part of the default run; or copy: a 512 MiB device copy used to calibrate the
rocprofv3 byte counters).
"""
import argparse
import ctypes as C
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

BYTES_PER_VOXEL_ITER = 84.0      # bytes of one max-flow iteration as two stencil passes
HBM_PEAK_GBS = 8000.0            # MI355X

# Algorithmic bytes of one pass of the multi-level sweep per voxel: each solve's
# state (hp x3, pt, tmp, u) read once and written once (48 B) and its alpha
# read (4 B), plus the fields a pass reads once for every solve it advances
# (frame as 4 floats, cs, ct: 24 B). A pass applies one to L iterations.
SWEEP_STATE_BYTES = 52.0
SWEEP_SHARED_BYTES = 24.0

# HBM bytes the same kernels moved per voxel-iteration, from rocprofv3 FETCH_SIZE
# and WRITE_SIZE passes scaled by a 512 MiB copy (FETCH_SIZE x 2.0, WRITE_SIZE x 1.0);
# the passes and their commands are recorded under profiles/
TRAFFIC_GRID_PER_VOXEL_ITER = 67.6     # batched p + u kernels, groups of 4 solves, 128^3
TRAFFIC_PLAIN_PER_VOXEL_ITER = 88.2    # per-iteration p + u kernels, 256^3
# the sweep by tile shape (1-based, as mh_cmf_sweep_choice reports it), one solve per
# thread, at 128^3 (two-level shapes) and at 256^3 (two, three and four levels)
TRAFFIC_SWEEP_PER_VOXEL_ITER = {1: 44.1, 2: 49.3, 3: 44.5, 4: 45.4, 5: 41.9}
TRAFFIC_SWEEP_256_PER_VOXEL_ITER = {1: 43.1, 2: 56.6, 3: 52.5, 4: 46.7, 5: 46.9, 6: 32.4, 7: 32.9,
                                    8: 27.6, 9: 28.0}
# the batched grid's sweep, two solves per thread (the 1024-thread tile shapes of
# two and three levels: 1, 4, 5, 6, 7), at 128^3, with the axial p-step: the two-level
# shape 1 and the three-level shape 7; shapes 4, 5 and 6 unmeasured
TRAFFIC_SWEEP_PAIR_PER_VOXEL_ITER = {1: 38.8, 7: 30.2}
PAIR_TILES = (1, 4, 5, 6, 7)
# iterations per pass of each tile shape (1-based)
SWEEP_LEVELS = {1: 2, 2: 2, 3: 2, 4: 2, 5: 2, 6: 3, 7: 3, 8: 4, 9: 4}
# Solves that stay on the chip (volumes of up to 2^21 voxels, the automatic method):
# vector instructions per voxel-iteration of the p- and the u-step with eigenvalues
# (l0, l1, l1), and the rate 256 compute units issue them at (64 lanes, 2.4 GHz);
# bytes per voxel and solve: u0, alpha, cs, ct and the frame in, u out
ONCHIP_VOXELS = 1 << 21
ONCHIP_INSTRUCTIONS = 74.0
VECTOR_ISSUE_T = 39.3
ONCHIP_BYTES_PER_VOXEL = 32.0
GRID_GROUP = 4                         # solves per group of the batched per-iteration kernels

PARTS = ("grid", "plain", "plain64", "plain256", "ragged", "serve", "cpu", "sigmas")


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def timed(torch, fn, reps=1):
    """Run fn reps times between HIP events on the current stream; returns seconds."""
    s = torch.cuda.current_stream()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    e0.record(s)
    for _ in range(reps):
        fn()
    e1.record(s)
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / 1e3


def sweep_choice(dev, shape, batched=False):
    """The tile shape (1-based) of the multi-level sweep the library tuned for
    volumes of this shape (with batched, the batched solver's pair choice when
    it made one), or 0 for the per-iteration kernels / not tuned."""
    from miccai2016_amd import _lib
    tile, zc = C.c_int(0), C.c_int(0)
    if batched:
        ok = dev.lib.mh_cmf_batched_sweep_choice(dev.handle, _lib.dims3(shape), C.byref(tile),
                                                 C.byref(zc))
        if ok == 1:
            return tile.value
    ok = dev.lib.mh_cmf_sweep_choice(dev.handle, _lib.dims3(shape), C.byref(tile), C.byref(zc))
    return tile.value if ok == 1 else 0


def sweep_passes(iters, update, levels=2):
    """Passes of an L-level sweep for a solve of `iters` iterations: a
    criterion iteration always ends its pass, and a pass stops short of
    the end."""
    it = passes = 0
    while it < iters:
        lv = 1
        while lv < levels and it + lv < iters and (it + lv - 1) % update != 0:
            lv += 1
        it += lv
        passes += 1
    return passes


def device_pipeline(dev, spec, weighting, decay, cfg, timings, seed=42):
    """A helix phantom generated on the device and the full preparation
    (Frangi, direction adjustment, GVF, frame completion, capacities) of its
    cut: (u0, frames, alpha, cs, ct, truth) device tensors; stage seconds go
    into `timings`."""
    from miccai2016_amd import _lib
    from miccai2016_amd.pipeline import prepare_device
    shape = spec.shape
    n = int(np.prod(shape))
    L, h, st = dev.lib, dev.handle, dev.stream
    img, truth = dev.empty(n), dev.empty(n, dtype=dev.torch.uint8)
    dev.check(L.mh_helix_phantom(h, _lib.dims3(shape), spec.r_tube, spec.r_helix, spec.pitch,
                                 spec.sigma, C.c_uint64(seed), dev.ptr(img), dev.ptr(truth), None,
                                 st), "mh_helix_phantom")
    prep = prepare_device(img, shape, spec.sigma, cfg, dev, timings=timings)
    al, u0 = dev.empty(n), dev.empty(n)
    dev.check(L.mh_nonterminal_weight(h, dev.ptr(prep.gms), n, weighting, decay, dev.ptr(al), st),
              "mh_nonterminal_weight")
    wk = dev.empty(int(L.mh_initial_u_work_floats(n)))
    dev.check(L.mh_initial_u(h, dev.ptr(img), n, dev.ptr(u0), dev.ptr(wk), st), "mh_initial_u")
    timings["ridge_voxels"] = prep.ridge_voxels
    return u0, prep.quats, al, prep.cs, prep.ct, truth


def _cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for ln in f:
                if ln.startswith("model name"):
                    return ln.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--iters", type=int, default=500, help="max-flow iterations per solve")
    ap.add_argument("--solves", type=int, default=425, help="grid cells per step (<= 425)")
    ap.add_argument("--plain-solves", type=int, default=6)
    ap.add_argument("--only", choices=PARTS + ("copy",), default=None)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-256", action="store_true")
    ap.add_argument("--no-serve", action="store_true")
    ap.add_argument("--iters-256", type=int, default=1000)
    ap.add_argument("--sweep", type=int, default=0,
                    help="multi-level sweep of single solves: 0 tuned, 1 off, 2 on")
    ap.add_argument("--sweep-tile", type=int, default=0,
                    help="with --sweep 2: the tile shape (1-5 two levels, 6-7 three, 8-9 "
                         "four; 0: the first)")
    ap.add_argument("--batched-sweep", type=int, default=0,
                    help="batched grid: 0 automatic, 1 per-iteration kernels of groups, 2 sweep")
    ap.add_argument("--cpu-iters", type=int, default=500)
    ap.add_argument("--cpu-solves", type=int, default=2, help="grid cells the CPU oracle solves")
    ap.add_argument("--serve-qps", type=str, default="5,10,20,40,80,160,200",
                    help="comma-separated arrival rates; one serving run each")
    ap.add_argument("--serve-seconds", type=float, default=4.0,
                    help="arrival span per rate: requests = rate x seconds, within "
                         "[--serve-min-requests, --serve-max-requests]")
    ap.add_argument("--serve-min-requests", type=int, default=20)
    ap.add_argument("--serve-max-requests", type=int, default=120)
    ap.add_argument("--serve-max-queue", type=int, default=48,
                    help="requests waiting for admission beyond which new ones are refused")
    ap.add_argument("--serve-pipeline-qps", type=str, default="2",
                    help="QPS of requests served through the full preparation ('' skips)")
    ap.add_argument("--serve-pipeline-requests", type=int, default=20)
    ap.add_argument("--serve-prepare-workers", type=int, default=4)
    ap.add_argument("--ragged-volumes", type=int, default=64)
    ap.add_argument("--sigmas", type=int, default=15,
                    help="noise levels of --only sigmas (the first of linspace(0.1, 1.5, 15))")
    ap.add_argument("--sigmas-no-tv", action="store_true",
                    help="--only sigmas runs the ATV grid only, not the TV grid beside it")
    ap.add_argument("--ragged-workers", type=int, default=8,
                    help="threads preparing the ragged volumes (own context and stream each)")
    ap.add_argument("--no-ragged", action="store_true")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the library has no multi-GPU path; the solver runs "
              "on one device (run with --gpus 1)", file=sys.stderr)
        sys.exit(2)
    run = {p: (args.only == p) if args.only else True for p in PARTS}
    if not args.only:
        run["cpu"] = not args.no_cpu
        run["sigmas"] = False      # the whole experiment: --only sigmas
        run["plain256"] = not args.no_256
        run["serve"] = not args.no_serve
        run["ragged"] = not args.no_ragged

    import torch
    from miccai2016_amd import phantom as ph
    from miccai2016_amd.device import default_context
    from miccai2016_amd.pipeline import PipelineConfig, cut_parameters, prepare
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import (
        CmfCutQAnisotropicGpu, initial_u)

    dev = default_context(0)
    dev.check(dev.lib.mh_cmf_set_sweep(dev.handle, args.sweep, args.sweep_tile, 0), "mh_cmf_set_sweep")
    dev.check(dev.lib.mh_cmf_batched_set_sweep(dev.handle, args.batched_sweep),
              "mh_cmf_batched_set_sweep")

    if args.only == "copy":
        a = torch.ones(128 << 20, device=dev.device)
        b = torch.empty_like(a)
        torch.cuda.synchronize()
        b.copy_(a)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes": a.numel() * 4}), flush=True)
        return

    cfg = PipelineConfig()
    cfg.cut_iters = args.iters
    eigs = (1, cfg.a_atv, cfg.a_atv)
    w_all, d_all = ph.grid_pairs()
    S = max(1, min(args.solves, len(w_all)))
    line = {
        "metric": "ATV max-flow voxel-iters/s, batched vs plain at Dice>=0.999; p50/p99 latency",
        "value": None, "unit": "voxel-iters/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": None, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic helix phantom (seeded)",
        "config": {"workload": f"batched grid search, {S} ATV solves x {args.iters} iterations "
                               f"on one 128^3 helix phantom (sigma 1.5)",
                   "solves": S, "iterations": args.iters, "volume": [128, 128, 128]},
    }

    if run["grid"] or run["plain"] or run["cpu"]:
        spec = ph.GRID_128
        log(f"phantom {spec.shape} sigma={spec.sigma}")
        img, truth = ph.make_helix(spec)
        t0 = time.time()
        prep = prepare(img, spec.sigma, cfg, dev)
        torch.cuda.synchronize()
        line["prepare_s"] = time.time() - t0
        log(f"prepare (Frangi, adjustment, GVF, frames, capacities): {line['prepare_s']:.2f} s")
        n = img.size
        q_d = dev.upload(prep.quats).reshape(-1)
        gms_d = dev.upload(prep.gms).reshape(-1)
        cs_d, ct_d = dev.upload(prep.cs).reshape(-1), dev.upload(prep.ct).reshape(-1)
        u0 = dev.upload(initial_u(img)).reshape(1, -1)

    # ---- the batched grid (the headline)
    ub = None
    if run["grid"]:
        w, d = w_all[:S].astype(np.float32), d_all[:S].astype(np.float32)
        cutter = CmfCutQAnisotropicGpu(cut_parameters(cfg), dev)
        u = torch.empty((S, n), dtype=torch.float32, device=dev.device)

        def step():
            u.copy_(u0.expand(S, n))
            cutter.execute_batched_device(u, S, w, d, q_d, gms_d, cs_d, ct_d, img.shape, eigs)

        for k in range(args.warmup):
            step()
            torch.cuda.synchronize()
            log(f"warmup step {k + 1}/{args.warmup} done")
        secs = 0.0
        done_iters = 0
        for k in range(args.steps):
            secs += timed(torch, step)
            # the iterations every solve actually ran (a NaN stop ends a solve early)
            done_iters += sum(int(r.iterations) for r in cutter.last_result)
            log(f"timed step {k + 1}/{args.steps}: {secs / (k + 1):.3f} s/step")
        value = float(done_iters) * n / secs
        line["value"] = value
        line["ms_per_step"] = secs / args.steps * 1e3
        line["config"]["iterations_run"] = done_iters // args.steps
        line["config"]["stopped_solves"] = sum(int(r.stopped != 0) for r in cutter.last_result)
        log(f"batched grid: {value:.4e} voxel-iters/s ({line['ms_per_step']:.1f} ms/step, "
            f"{done_iters // args.steps} solve-iterations per step)")
        from miccai2016_amd.evaluation import DeviceDice
        grid_dice = DeviceDice(truth, dev)(u, S)
        best = int(np.nanargmax(grid_dice))
        from miccai2016_amd.evaluation import device_dice_for
        true_dice, _ = device_dice_for(u[best], truth, img.shape, dev)
        line["grid_quality"] = {"best_fast_dice": float(grid_dice[best]),
                                "dice_of_largest_component": float(true_dice),
                                "best_weighting": float(w_all[best]),
                                "best_decay": float(d_all[best])}
        log(f"grid: best fast Dice {grid_dice[best]:.4f} at w={w_all[best]:.4g}, "
            f"decay={d_all[best]:.4g}")
        tile = sweep_choice(dev, img.shape, batched=True)
        if args.sweep == 2 and args.batched_sweep != 1:
            tile = args.sweep_tile or 1      # forced, not tuned
        step_s = secs / args.steps
        effective = value * BYTES_PER_VOXEL_ITER / 1e9
        if args.sweep == 0 and args.batched_sweep == 0 and n <= ONCHIP_VOXELS:
            # solve after solve in the registers of one launch (the first two
            # through the sweep where the pair tuner still had to time it)
            achieved = value * ONCHIP_INSTRUCTIONS / 1e12
            line["roofline"] = {
                "bound": "vector issue", "achieved": achieved, "peak": VECTOR_ISSUE_T,
                "unit": "T lane-instructions/s", "frac": achieved / VECTOR_ISSUE_T,
                "traffic": ONCHIP_BYTES_PER_VOXEL * n * S,
                "kernel": f"cmf_onchip_kernel: one launch = {S} solves of {args.iters} max-flow "
                          "iterations, the state in registers, brick faces as tagged words",
                "algorithmic": f"{ONCHIP_INSTRUCTIONS:.0f} vector instructions per "
                               "voxel-iteration (p-step 47, u-step 27)",
                "us_per_iteration": step_s / (S * args.iters) * 1e6,
                "algorithmic_hbm_GBs": ONCHIP_BYTES_PER_VOXEL * n * S / step_s / 1e9,
                "effective_GBs_84B": effective,
                "effective_frac_84B": effective / HBM_PEAK_GBS}
        elif tile:
            # the groups ran one after another through the multi-level sweep:
            # one launch is one pass of up to L iterations over a pair of
            # solves (the 1024-thread tile shapes of up to three levels) or
            # over one solve
            levels = SWEEP_LEVELS.get(tile, 2)
            passes = sweep_passes(args.iters, cfg.cut_update, levels)
            pair = tile in PAIR_TILES and n < (1 << 26)
            per_launch = 2 if pair else 1
            launches = (S // per_launch + S % per_launch) * passes
            pass_bytes = (per_launch * SWEEP_STATE_BYTES + SWEEP_SHARED_BYTES) * n
            step_bytes = (S // per_launch) * passes * pass_bytes
            if S % per_launch:
                step_bytes += passes * (SWEEP_STATE_BYTES + SWEEP_SHARED_BYTES) * n
            achieved = step_bytes / step_s / 1e9
            per_vi = (TRAFFIC_SWEEP_PAIR_PER_VOXEL_ITER if pair
                      else TRAFFIC_SWEEP_PER_VOXEL_ITER).get(tile)
            line["roofline"] = {
                "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": achieved / HBM_PEAK_GBS,
                "traffic": None if per_vi is None else per_vi * levels * per_launch * n,
                "kernel": f"{'cmf_sweep_kernel' if levels == 2 else 'cmf_sweepL_kernel'} (tile "
                          f"shape {tile}, {per_launch} solve(s) per thread): one launch = one pass "
                          f"of up to {levels} max-flow iterations over {per_launch} solve(s)",
                "algorithmic_bytes_per_launch": pass_bytes,
                "algorithmic_bytes": "the blocked scheme's minimum: per pass and voxel, each "
                                     "solve's state (hp x3, pt, tmp, u) read and written once and "
                                     "its alpha read (52 B), the frame (16 B) and cs, ct read once "
                                     "for the pair",
                "launch_us": step_s / launches * 1e6,
                "traffic_per_voxel_iteration": per_vi,
                # the measured bytes over the same launches, beside the
                # scheme's minimum that `achieved` and `frac` take
                "achieved_traffic_GBs": None if per_vi is None else per_vi * value / 1e9,
                "frac_traffic": None if per_vi is None else per_vi * value / 1e9 / HBM_PEAK_GBS,
                "traffic_note": f"measured HBM bytes per launch of {levels} iterations "
                                "(rocprofv3 FETCH_SIZE x 2.0 + WRITE_SIZE, copy-calibrated); at "
                                "128^3 one pair's working set (~250 MB) mostly stays in the 256 "
                                "MB last-level cache",
                "effective_GBs_84B": effective,
                "effective_frac_84B": effective / HBM_PEAK_GBS}
        else:
            groups = -(-S // GRID_GROUP)
            achieved = effective
            line["roofline"] = {
                "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": achieved / HBM_PEAK_GBS,
                "traffic": TRAFFIC_GRID_PER_VOXEL_ITER * GRID_GROUP * n,
                "kernel": "one max-flow iteration of a group of 4 solves: cmf_batch_p_kernel<4> + "
                          "cmf_batch_u_kernel<4> (84 algorithmic B per solve-voxel-iteration; "
                          "traffic = measured HBM bytes per such launch pair)",
                "launch_us": step_s / (groups * args.iters) * 1e6,
                "traffic_per_voxel_iteration": TRAFFIC_GRID_PER_VOXEL_ITER}
        ub = u.detach().cpu().numpy()
        del u

    # ---- the same solves one at a time (device-resident) and through the API
    if run["plain"]:
        P = max(1, min(args.plain_solves, S))
        pick = np.linspace(0, S - 1, P).astype(int)
        plain_cut = CmfCutQAnisotropicGpu(cut_parameters(cfg), dev)
        alphas = [ph.nonterminal_weight(prep.gms, w_all[j], d_all[j]).astype(np.float32)
                  for j in pick]
        ud = dev.empty(n)
        t_dev, dices = 0.0, []
        for j, a in zip(pick, alphas):
            a_d = dev.upload(a).reshape(-1)

            def one():
                ud.copy_(u0.reshape(-1))
                plain_cut.execute_device(ud, q_d, a_d, cs_d, ct_d, const_sqevals=np.sqrt(eigs),
                                         shape=img.shape)
            one()          # the first solve of a shape runs the default method,
            one()          # the second tunes it (unless the grid's probe did)
            t_dev += timed(torch, one)
            if ub is not None:
                dices.append(ph.dice_between(ub[j], ud.detach().cpu().numpy()))
        per_dev = t_dev / P
        t_api = 0.0
        napi = min(P, 3)
        for j, a in zip(pick[:napi], alphas[:napi]):
            t1 = time.time()
            plain_cut.execute(img, prep.quats, eigs, a, prep.cs, prep.ct, verbose=False)
            t_api += time.time() - t1
        per_api = t_api / napi
        plain_rate = n * args.iters / per_dev
        line["plain"] = {"voxel_iters_per_s": plain_rate, "ms_per_solve_device": per_dev * 1e3,
                         "ms_per_solve_numpy_api": per_api * 1e3,
                         "sequential_425_s_device": per_dev * 425,
                         "sequential_425_s_numpy_api": per_api * 425}
        if line["value"]:
            line["plain"].update(
                batched_speedup_vs_device=line["value"] / plain_rate,
                batched_speedup_vs_numpy_api=line["value"] / (n * args.iters / per_api),
                min_dice_batched_vs_plain=float(min(dices)))
        log(f"plain device-resident: {per_dev * 1e3:.2f} ms/solve; numpy API: "
            f"{per_api * 1e3:.2f} ms/solve")

    # ---- 64^3 single solve through the whole pipeline (the reference's own case)
    if run["plain64"]:
        from miccai2016_amd.evaluation import DeviceDice, device_dice_for
        spec = ph.PLAIN_64
        # the first run in the process pays one-time costs (code-object loads,
        # host thread pools); the second is the pipeline's own time
        t0 = time.perf_counter()
        device_pipeline(dev, spec, 10 ** -1.625, 10 ** 1.5, cfg, {})
        torch.cuda.synchronize()
        t_cold = time.perf_counter() - t0
        prep64 = {}
        t0 = time.perf_counter()
        u0s, qs, als, css, cts, trs = device_pipeline(dev, spec, 10 ** -1.625, 10 ** 1.5, cfg,
                                                      prep64)
        t_prep = time.perf_counter() - t0
        us = torch.empty_like(u0s)
        c64 = CmfCutQAnisotropicGpu(cut_parameters(cfg), dev)

        def solve64():
            us.copy_(u0s)
            c64.execute_device(us, qs, als, css, cts, const_sqevals=np.sqrt(eigs),
                               shape=spec.shape)
        solve64()          # the first solve of a shape runs the default method,
        solve64()          # the second tunes it
        t64 = timed(torch, solve64)
        n64 = u0s.numel()
        try:
            dice64, _ = device_dice_for(us, trs, spec.shape, dev)
        except ValueError:          # an empty cut
            dice64 = float("nan")
        line["plain_64"] = {
            "pipeline_s": t_prep + t64, "first_prepare_in_process_s": t_cold,
            "prepare_s": {k: v for k, v in prep64.items()
                                                      if k != "ridge_voxels"},
            "ridge_voxels": prep64["ridge_voxels"], "solve_ms": t64 * 1e3,
            "iterations": cfg.cut_iters, "voxel_iters_per_s": n64 * cfg.cut_iters / t64,
            "fast_dice_vs_truth": float(DeviceDice(trs, dev)(us, 1)[0]),
            "dice_of_largest_component": float(dice64),
            "workload": "64^3 helix (tube 4, radius 16, pitch 24, noise 1.5): Frangi (3 scales), "
                        "adjustment, GVF (200 iterations), 500 ATV max-flow iterations"}
        log(f"64^3 pipeline: prepare {prep64}, solve {t64 * 1e3:.1f} ms, Dice "
            f"{line['plain_64']['fast_dice_vs_truth']:.4f}")
        del u0s, qs, als, css, cts, trs, us

    # ---- 256^3 single solve (bandwidth scale)
    if run["plain256"]:
        spec = ph.PLAIN_256
        it256 = args.iters_256
        prep256 = {}
        u0b, qb, al_b, cs_b, ct_b, tr_b = device_pipeline(dev, spec, 10 ** -1.625, 10 ** 1.5, cfg,
                                                          prep256)
        nb = u0b.numel()
        ub_ = torch.empty(nb, device=dev.device)
        p256 = cut_parameters(cfg)
        p256.num_iter = it256
        c256 = CmfCutQAnisotropicGpu(p256, dev)

        def solve256():
            ub_.copy_(u0b)
            c256.execute_device(ub_, qb, al_b, cs_b, ct_b, const_sqevals=np.sqrt(eigs),
                                shape=spec.shape)
        solve256()         # the first solve of a shape runs the default method,
        solve256()         # the second tunes it
        t256 = timed(torch, solve256)
        rate256 = nb * it256 / t256
        tile256 = sweep_choice(dev, spec.shape)
        line["plain_256"] = {"voxel_iters_per_s": rate256, "ms_per_solve": t256 * 1e3,
                             "iterations": it256, "sweep_tile": tile256,
                             "achieved_GBs_algorithmic": rate256 * BYTES_PER_VOXEL_ITER / 1e9,
                             "frac_algorithmic": rate256 * BYTES_PER_VOXEL_ITER / 1e9 / HBM_PEAK_GBS,
                             "traffic_per_voxel_iteration_sweep":
                                 TRAFFIC_SWEEP_256_PER_VOXEL_ITER.get(tile256),
                             "traffic_per_voxel_iteration_plain_kernels":
                                 TRAFFIC_PLAIN_PER_VOXEL_ITER}
        from miccai2016_amd.evaluation import DeviceDice
        line["plain_256"]["prepare_s"] = {k: v for k, v in prep256.items() if k != "ridge_voxels"}
        line["plain_256"]["ridge_voxels"] = prep256["ridge_voxels"]
        line["plain_256"]["fast_dice_vs_truth"] = float(DeviceDice(tr_b, dev)(ub_, 1)[0])
        log(f"256^3 x {it256} iterations: {t256:.3f} s -> {rate256:.4e} voxel-iters/s; "
            f"preparation {prep256}")
        del qb, al_b, cs_b, ct_b, u0b, ub_, tr_b

    # ---- ragged set: the full pipeline per volume, one packed max-flow solve
    if run["ragged"]:
        from miccai2016_amd import _lib
        from miccai2016_amd.evaluation import DeviceDice
        from miccai2016_amd.pipeline import segment_ragged
        specs, rw, rd = ph.ragged_set(args.ragged_volumes, seed=2016)
        vols, truths = [], []
        for sp in specs:
            nv = int(np.prod(sp.shape))
            im, tr = dev.empty(nv), dev.empty(nv, dtype=torch.uint8)
            dev.check(dev.lib.mh_helix_phantom(dev.handle, _lib.dims3(sp.shape), sp.r_tube,
                                               sp.r_helix, sp.pitch, sp.sigma,
                                               C.c_uint64(sp.seed), dev.ptr(im), dev.ptr(tr),
                                               None, dev.stream), "mh_helix_phantom")
            vols.append((im, sp.shape))
            truths.append(tr)
        rcfg = PipelineConfig()
        rcfg.cut_iters = args.iters
        rr = segment_ragged(vols, [sp.sigma for sp in specs], rw, rd, rcfg, dev,
                            workers=args.ragged_workers)
        total = int(sum(np.prod(sp.shape) for sp in specs))
        dice = [float(DeviceDice(tr, dev)(rr.volume(v).reshape(-1), 1)[0])
                for v, tr in enumerate(truths)]
        line["ragged"] = {
            "volumes": len(specs), "total_voxels": total, "iterations": args.iters,
            "prepare_s": rr.prepare_s, "prepare_workers": args.ragged_workers,
            "solve_s": rr.solve_s,
            "voxel_iters_per_s": total * args.iters / rr.solve_s,
            "median_fast_dice_vs_truth": float(np.nanmedian(dice)),
            "workload": "dims U[48,192] per axis, tube U[3,8], helix radius min(dims)/4, pitch "
                        "U[20,80], noise U[0.1,1.5], (w, decay) from the grid; Frangi, adjustment "
                        "and GVF per volume, one ragged max-flow solve (volumes of >= 2^19 voxels "
                        "one at a time through the tuned method, the rest packed)"}
        log(f"ragged: {len(specs)} volumes, {total} voxels, prepare {rr.prepare_s:.2f} s, "
            f"solve {rr.solve_s:.3f} s")
        del vols, truths, rr

    # ---- serving: Poisson arrivals of synthetic helix cuts of mixed sizes
    if run["serve"]:
        from miccai2016_amd.serving import MaxFlowServer, poisson_load, synthetic_request
        torch.cuda.empty_cache()
        line["serving"] = []
        runs = [(float(q), False,
                 int(min(args.serve_max_requests,
                         max(args.serve_min_requests, round(float(q) * args.serve_seconds)))))
                for q in args.serve_qps.split(",") if q]
        runs += [(float(q), True, args.serve_pipeline_requests)
                 for q in args.serve_pipeline_qps.split(",") if q]
        for qps, full, nreq in runs:
            srv = MaxFlowServer(cut_parameters(cfg), chunk=50,
                                prepare_workers=args.serve_prepare_workers,
                                max_queue=None if full else args.serve_max_queue).start()
            log(f"serving {nreq} {'prepared ' if full else ''}requests at {qps} QPS "
                f"(budget {srv.budget / 2 ** 30:.1f} GiB)")
            tickets = poisson_load(srv, lambda rng: synthetic_request(rng, prepare=full), qps,
                                   nreq, seed=11)
            srv.stop(drain=True, timeout=600)
            st = srv.stats()
            dice = [t.dice for t in tickets if t.dice is not None and not np.isnan(t.dice)]
            line["serving"].append({
                "qps": qps, "requests": nreq, "completed": st["completed"],
                "rejected_queue_full": st["rejected"], "max_queue": srv.max_queue,
                "peak_queue": st["peak_queue"], "queue_wait_p99_s": st.get("queue_wait_p99_s"),
                "errors": sum(t.error is not None for t in tickets) - st["rejected"],
                "p50_s": st.get("p50_s"), "p99_s": st.get("p99_s"), "mean_s": st.get("mean_s"),
                "voxel_iters_per_s": st.get("voxel_iters_per_s"),
                "offered_voxel_iters_per_s": qps * float(np.mean(
                    [np.prod(t.request.shape) * t.request.num_iter for t in tickets])),
                "peak_resident_jobs": srv.peak_resident,
                "peak_reserved_GiB": srv.peak_reserved / 2 ** 30,
                "budget_GiB": srv.budget / 2 ** 30, "chunk": srv.chunk,
                "median_dice_vs_truth": float(np.median(dice)) if dice else None,
                "frames": ("full preparation (Frangi, adjustment, GVF, completion) on "
                           f"{args.serve_prepare_workers} workers" if full
                           else "the phantom's centre-line frames"),
                "workload": "side log-U[64,320], aspect <= 2:1, 300-1000 iterations, helix/noise "
                            "as the ragged set, (w, decay) from the grid; cuts of >= 2^20 voxels "
                            "as resident solves, smaller ones as packed jobs"})
            log(f"serving at {qps} QPS: p50 {st.get('p50_s', 0):.3f} s, p99 {st.get('p99_s', 0):.3f} s,"
                f" {st.get('voxel_iters_per_s') or 0:.3e} voxel-iters/s, peak {srv.peak_resident} "
                f"resident, {st['rejected']} refused")
            del srv, tickets
            torch.cuda.empty_cache()   # the next server's budget starts from the free memory
        sweep = [r for r in line["serving"] if not r["frames"].startswith("full")]
        if sweep:
            # capacity: the most this workload was served at; saturation: the
            # first rate whose served throughput fell below 90 % of the offered
            cap = max((r["voxel_iters_per_s"] or 0.0) for r in sweep)
            sat = next((r["qps"] for r in sweep
                        if (r["voxel_iters_per_s"] or 0.0) < 0.9 * r["offered_voxel_iters_per_s"]
                        or r["rejected_queue_full"]), None)
            line["serving_summary"] = {
                "capacity_voxel_iters_per_s": cap, "saturation_qps": sat,
                "mean_request_voxel_iters": float(np.mean(
                    [r["offered_voxel_iters_per_s"] / r["qps"] for r in sweep])),
                "beyond_saturation": "arrivals beyond capacity queue up to max_queue and later "
                                     "ones are refused at submission (OverloadError), so p99 of "
                                     "the served requests stays bounded"}

    # ---- the experiment's grid at every noise level (all 15 noise levels)
    if run["sigmas"]:
        from miccai2016_amd import _lib
        from miccai2016_amd.evaluation import DeviceDice, device_dice_for
        from miccai2016_amd.pipeline import prepare_device
        w, d = w_all[:S].astype(np.float32), d_all[:S].astype(np.float32)
        base = ph.GRID_128
        shape = base.shape
        n = int(np.prod(shape))
        cutter = CmfCutQAnisotropicGpu(cut_parameters(cfg), dev)
        u = torch.empty((S, n), dtype=torch.float32, device=dev.device)
        rows, t_all = [], time.perf_counter()
        for sigma in np.linspace(0.1, 1.5, 15)[:max(1, args.sigmas)]:
            t0 = time.perf_counter()
            img, truth = dev.empty(n), dev.empty(n, dtype=torch.uint8)
            dev.check(dev.lib.mh_helix_phantom(dev.handle, _lib.dims3(shape), base.r_tube,
                                               base.r_helix, base.pitch, float(sigma),
                                               C.c_uint64(42), dev.ptr(img), dev.ptr(truth), None,
                                               dev.stream), "mh_helix_phantom")
            prep = prepare_device(img, shape, float(sigma), cfg, dev)
            u0 = dev.empty(n)
            wk = dev.empty(int(dev.lib.mh_initial_u_work_floats(n)))
            dev.check(dev.lib.mh_initial_u(dev.handle, dev.ptr(img), n, dev.ptr(u0), dev.ptr(wk),
                                           dev.stream), "mh_initial_u")
            dev.synchronize()
            t_prep = time.perf_counter() - t0

            def grid(eg):
                def grid_step():
                    u.copy_(u0.reshape(1, -1).expand(S, n))
                    cutter.execute_batched_device(u, S, w, d, prep.quats, prep.gms, prep.cs,
                                                  prep.ct, shape, eg)
                t_grid = timed(torch, grid_step)
                fd = DeviceDice(truth, dev)(u, S)
                best = int(np.nanargmax(fd))
                try:
                    true_dice = float(device_dice_for(u[best], truth, shape, dev)[0])
                except ValueError:
                    true_dice = float("nan")
                return {"grid_s": t_grid, "voxel_iters_per_s": S * n * args.iters / t_grid,
                        "best_fast_dice": float(fd[best]), "dice_of_largest_component": true_dice,
                        "best_weighting": float(w_all[best]), "best_decay": float(d_all[best])}

            row = {"sigma": float(sigma), "prepare_s": t_prep, "ridge_voxels": prep.ridge_voxels}
            row.update(grid(eigs))
            msg = (f"sigma {sigma:.2f}: prepare {t_prep:.2f} s, ATV grid {row['grid_s']:.2f} s, "
                   f"best fast Dice {row['best_fast_dice']:.4f} (largest component "
                   f"{row['dice_of_largest_component']:.4f}) at w={row['best_weighting']:.4g}, "
                   f"decay={row['best_decay']:.4g}")
            if not args.sigmas_no_tv:
                # the experiment's second regularisation: isotropic TV, eigenvalues (1, 1, 1)
                # (phantom_experiment.py:365-368)
                row["tv"] = grid((1.0, 1.0, 1.0))
                tv = row["tv"]
                msg += (f"; TV grid {tv['grid_s']:.2f} s, best fast Dice {tv['best_fast_dice']:.4f}"
                        f" (largest component {tv['dice_of_largest_component']:.4f}) at "
                        f"w={tv['best_weighting']:.4g}, decay={tv['best_decay']:.4g}")
            rows.append(row)
            log(msg)
            del prep, img, truth, u0
        line["grid_sigmas"] = {
            "levels": rows, "total_s": time.perf_counter() - t_all,
            "workload": f"{S} ATV solves{'' if args.sigmas_no_tv else f' and {S} TV solves'} x "
                        f"{args.iters} iterations per noise level on the 128^3 helix "
                        "(tube 6, radius 32, pitch 48), noise linspace(0.1, 1.5, 15); Frangi, "
                        "adjustment and GVF once per level on the device"}
        del u

    # ---- CPU oracle on a bounded sample of the same workload, and the
    # oracle's results beside the GPU's on the same inputs
    if run["cpu"]:
        from oracle import chain, ref32
        try:
            build_flags = ref32.use_native_build()
        except Exception as e:          # no compiler: the portable build is timed
            build_flags = f"portable x86-64-v3 build (native build failed: {e})"
        threads = len(os.sched_getaffinity(0))
        ref32.set_num_threads(threads)
        ncpu = max(1, min(args.cpu_solves, len(w_all)))
        # the reference's own best cell (w 10^-1.625, decay 10^1.5) first, then
        # the grid's best cell in this run, then cells in grid order
        cells = [int(np.argmin(np.abs(np.log10(w_all) + 1.625) + np.abs(np.log10(d_all) - 1.5)))]
        if "grid_quality" in line:
            cells.append(int(np.argmin(np.abs(w_all - line["grid_quality"]["best_weighting"]) +
                                       np.abs(d_all - line["grid_quality"]["best_decay"]))))
        cells += [j for j in range(len(w_all)) if j not in cells]
        cells = [j for j in dict.fromkeys(cells) if j < S][:ncpu]
        parity = []
        tc = 0.0
        for j in cells:
            a0 = ph.nonterminal_weight(prep.gms, w_all[j], d_all[j]).astype(np.float32)
            t1 = time.time()
            uo, done, _ = ref32.cmf_solve(img, prep.quats, eigs, a0, prep.cs, prep.ct,
                                          steps=cfg.steps, cc=cfg.cc, num_iter=args.cpu_iters,
                                          update=cfg.cut_update, error_bound=0)
            tc += time.time() - t1
            if ub is not None and args.cpu_iters == args.iters:
                parity.append({"cell": j, "weighting": float(w_all[j]), "decay": float(d_all[j]),
                               "max_abs_u": float(np.abs(ub[j].reshape(img.shape) - uo).max()),
                               "dice_cut": float(ph.dice_between(ub[j].reshape(img.shape), uo)),
                               "iterations": int(done)})
        line["cpu_baseline"] = {
            "value": len(cells) * n * args.cpu_iters / tc, "unit": "voxel-iters/s",
            "cores": threads, "kind": "port", "cpu_model": _cpu_model(), "build": build_flags,
            "sample": f"{len(cells)} of the 425 solves, {args.cpu_iters} of 500 iterations each, "
                      f"128^3: CPU restatement (reference algorithm), C/OpenMP ({tc:.1f} s)"}
        if parity:
            line["parity_grid_cells"] = parity
            log("oracle vs GPU grid cells: " + ", ".join(
                f"cell {p['cell']}: max|du| {p['max_abs_u']:.2e}, Dice {p['dice_cut']:.6f}"
                for p in parity))
        log(f"cpu oracle: {line['cpu_baseline']['value']:.4e} voxel-iters/s on {threads} threads")
        # the 64^3 workload end to end: the oracle's chain (every stage) against
        # the GPU pipeline through the numpy API, and the CPU time of each
        spec = ph.PLAIN_64
        img64, truth64 = ph.make_helix(spec)
        w64, d64 = 10 ** -1.625, 10 ** 1.5
        t1 = time.time()
        cprep = chain.prepare(img64, spec.sigma)
        t2 = time.time()
        u_or, _ = chain.cut(img64, cprep, w64, d64)
        t3 = time.time()
        gprep = prepare(img64, spec.sigma, cfg, dev)
        from miccai2016_amd.pipeline import segment
        u_gpu = segment(img64, gprep, w64, d64, cfg, dev)
        line["cpu_baseline"]["plain_64"] = {
            "voxel_iters_per_s": img64.size * 500 / (t3 - t2), "solve_s": t3 - t2,
            "pipeline_s": t3 - t1, "prepare_s": t2 - t1,
            "sample": "the whole 64^3 workload on the CPU restatement: Frangi (3 scales), "
                      "adjustment, GVF (200), frames, 500 max-flow iterations"}
        line["parity_pipeline_64"] = {
            "max_abs_u": float(np.abs(u_gpu - u_or).max()),
            "dice_cut": float(ph.dice_between(u_gpu, u_or)),
            "fast_dice_vs_truth_gpu": float(ph.fast_dice(u_gpu, truth64)),
            "fast_dice_vs_truth_oracle": float(ph.fast_dice(u_or, truth64)),
            "oracle_ridge": cprep.info,
            "note": "every stage on both sides (oracle chain: ref32 kernels, scipy labelling, "
                    "the host spanning tree shared); GPU: prepare + segment. Across the tube "
                    "l2 ~ l3, so the ridge test's (v2, v3) plane is fixed but not its axes; FP32 "
                    "differences turn them and move ridge voxels, which at these small Frangi "
                    "scales flips whole branches: the cuts agree statistically (Dice vs truth), "
                    "and stage by stage exactly (parity_pipeline_64_staged)"}
        log(f"64^3 pipeline, oracle vs GPU: {line['parity_pipeline_64']}")
        # stage by stage: the GPU's adjustment from the oracle's ridge candidates
        # and main directions, then GVF, frames and cut from the oracle's directions
        from miccai2016_amd.processing.adjust_directions import (AdvancedAdjuster,
                                                                 TransformationCompleter)
        from miccai2016_amd.processing.gradient_vector_flow import GvfGpu, GvfParameters
        ves32 = cprep.vesselness.astype(np.float32)
        cand_o = ref32.detect_ridges(ves32, cprep.qeig, cfg.ridge_thresholds[0]) != 0
        adj = AdvancedAdjuster(cfg.ridge_thresholds, None, None, cfg.voxel_size, loader=dev)
        dirs_t = adj.execute_tensor(
            None, dev.upload(ves32).reshape(-1), img64.shape,
            candidates_t=dev.upload(cand_o.astype(np.float32)).reshape(-1),
            main_dirs_t=dev.upload(ref32.main_dirs(cprep.qeig)).reshape(-1))
        dirs_g = dev.download(dirs_t).reshape(img64.shape + (3,))
        gp = GvfParameters()
        gp.mu, gp.tol, gp.maxiter = cfg.gvf_mu, 0, cfg.gvf_iters
        gp.callback, gp.update, gp.normalize = None, max(cfg.gvf_iters // 10, 1), False
        v_or = (cprep.dirs.astype(np.float64) * cprep.vesselness[..., None]).astype(np.float32)
        q_or = TransformationCompleter(GvfGpu(v_or, gp, cfg.voxel_size,
                                              cl_program_loader=dev).execute(), dev).complete()
        gprep.quats, gprep.cs, gprep.ct = q_or, cprep.cs, cprep.ct
        u_st = segment(img64, gprep, w64, d64, cfg, dev)
        line["parity_pipeline_64_staged"] = {
            "ridge_voxels_differing": int((np.asarray(adj.ridge, bool) != cprep.ridge).sum()),
            "directions_bit_identical": bool(np.array_equal(dirs_g, cprep.dirs)),
            "adjustment_form": "device" if adj.device_used else "host",
            "cut_from_oracle_directions": {"max_abs_u": float(np.abs(u_st - u_or).max()),
                                           "dice_cut": float(ph.dice_between(u_st, u_or))},
            "note": "GPU adjustment from the oracle's ridge candidates and main directions; GPU "
                    "GVF, frames and cut from the oracle's adjusted directions"}
        log(f"64^3 pipeline stage by stage: {line['parity_pipeline_64_staged']}")

    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
