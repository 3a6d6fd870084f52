"""Benchmark: MLUPS of the coupled D3Q27 HOME step on one MI355X.

Workload: the 256x128x128 HOME dam break with four seeded 16-cell ice cubes
(``projecticy_amd.iceflow3d.workloads.dam_break_four_ice``), FP32, the full
coupled step (phase AA collide, forces, HOME collide/stream, recovery,
gradients, host rigid bodies, geometry refresh/refill, heat advection and
the 8-step conduction/melt update).  MLUPS = nx*ny*nz*steps/seconds/1e6 over
all cells, the reference's own definition.

The JSON line adds:
  roofline      the dominant kernel group of the flow step: algorithmic HBM
                bytes per launch / its mean duration (HIP events on the
                solver stream, a profiled pass after the timed region),
                against the 8 TB/s MI355X HBM peak, with the counted HBM
                bytes and the counted VALU busy fraction beside it;
  cpu_baseline  the FP64 C oracle (OpenMP on the host's cores, thread count
                and CPU model stated) on 8 steps of the same workload
                (including one conduction/melt update);
  d2q9          the coupled D2Q9 step on the 1024x2048 falling-ice case
                (FP32 populations, FP64 thermal), timed after the headline,
                with its own CPU baseline (the 2D oracle on 8 steps of the
                same case);
  ensemble      64 uneven D2Q9 cases (widths 64-512) stepped as one batch
                (one launch per kernel for all cases) with FP16 momentum
                (stochastic rounding; the headline storage), FP32 and
                all-FP16 (phase populations stored relative to w_q*phi)
                population storage: cases/hour for 10,000-step cases, the
                same figure for one-case-at-a-time FP32 runs, and the
                fine-solver gate: one case per width run 10,000 steps in
                each storage against the same case on a twice finer grid
                (FP32, 20,000 steps); ``value`` counts only the cases whose
                width melts within 1% of the fine solver;
  closure       the learned closure's BF16 MFMA forward and backward kernels
                on the 128x64x64 coarse grid, in TFLOP/s against the 2.5
                PFLOP/s dense BF16 peak.
"""

import argparse
import json
import math
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0
# Algorithmic bytes per cell of each flow-step kernel group: every field the
# group must read or write once (FP32 = 4 B, labels 1 B), neighbour reuse free.
KERNEL_BYTES = {
    "phase_collide": 4 * (7 + 1 + 3 + 3) + 1 + 4 * (7 + 3),          # h, phi, u, grad, id -> h, flux
    "forces": 4 * (1 + 3 + 3 + 3 + 1 + 2) + 2 + 4 * 6,             # phi, grad, u, flux, p*, V,E, labels -> F, a
    "home_collide_stream": 4 * (10 + 3 + 3) + 2 + 4 * (10 + 3),      # home, a, phi, V,E, labels -> home, u
    "phase_recover": 4 * (7 + 1 + 3) + 1 + 4 * 3,                    # h, p*, u, id -> h0, phi, p
    "gradients": 4 * 1 + 2 + 4 * 3,                                  # phi, labels -> grad
}
STEP_BYTES = 161  # minimal persistent state per cell-update of the whole step
# Counted HBM bytes and VALU busy of each kernel group, written by
# profile_counters.py from rocprofv3 counter runs of this script (the command
# is in the summary's .md beside it).  Used only while the kernel sources
# still hash to the value recorded there.
COUNTERS = ROOT / "profiles" / "counters_dam_break_256x128x128.json"
COUNTERS_2D = ROOT / "profiles" / "counters_d2q9_falling_ice_1024x2048.json"
# The 2D fused collide-stream's algorithmic bytes per cell (FP32 populations):
# f, h, phi, u, p, FP64 water volume and energy (the temperature), the label
# read; f, h, phi, u, a and the population sum written.
D2Q9_FUSED_BYTES = 4 * (9 + 9 + 1 + 2 + 1) + 8 * 2 + 1 + 4 * (9 + 9 + 1 + 2 + 2 + 1)


def measured_counters(path=COUNTERS, workload="dam_break"):
    """(summary, None) when the counter summary matches the current kernel
    sources, else (None, reason)."""
    if not path.exists():
        return None, "no counter summary"
    from profile_counters import source_hash

    data = json.loads(path.read_text())
    current = source_hash(workload)
    if data.get("source_sha") != current:
        return None, f"stale: counters taken on sources {data.get('source_sha')}, now {current}"
    return data, None


def copy_bandwidth(mib=1024, repeats=10):
    """Device-to-device copy bandwidth (bytes read + written per second) of
    torch's copy kernel over ``mib`` MiB, timed with HIP events."""
    import torch

    src = torch.ones(mib * (1 << 18), dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    dst.copy_(src)
    stream = torch.cuda.current_stream()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for _ in range(repeats):
        dst.copy_(src)
    end.record(stream)
    end.synchronize()
    seconds = start.elapsed_time(end) / 1e3 / repeats
    del src, dst
    return 2.0 * mib * (1 << 20) / seconds / 1e9


def parse():
    p = argparse.ArgumentParser(description=__doc__)
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=1000)
    p.add_argument("--warmup", type=int, default=20)
    p.add_argument("--profile-steps", type=int, default=64)
    p.add_argument("--seed", type=int, default=2026)
    p.add_argument("--size", type=int, nargs=3, default=(256, 128, 128))
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--d2q9-steps", type=int, default=200,
                   help="steps of the 1024x2048 D2Q9 case timed after the headline (0 skips it)")
    p.add_argument("--copy-probe-mib", type=int, default=0,
                   help="after the measurements, run five FP32 scale-by-one copies of this many MiB (the "
                        "reference kernel for calibrating HBM byte counters)")
    p.add_argument("--closure-repeats", type=int, default=20,
                   help="timed forward+backward passes of the closure network at 128x64x64 (0 skips it)")
    p.add_argument("--curve-steps", type=int, default=0,
                   help="also run the 3D workload from its initialisation for this many steps, timing each "
                        "100-step window (the ms-per-step curve over the full run)")
    p.add_argument("--curve-md", type=Path, default=None, help="write the curve as a Markdown table here")
    p.add_argument("--closure-score-steps", type=int, default=4096,
                   help="coarse steps of the closure's halved dam-break trajectory (0 to skip)")
    p.add_argument("--ensemble-cases", type=int, default=64)
    p.add_argument("--ensemble-steps", type=int, default=400,
                   help="timed steps of the batched FP16 D2Q9 ensemble (0 skips it)")
    p.add_argument("--ensemble-gate-steps", type=int, default=10000,
                   help="coarse steps of the fine-solver gate: one case per width in every storage against the "
                        "same case on a twice finer grid over the same physical time (0 skips it)")
    return p.parse_args()


D2Q9_STEP_BYTES = 185  # two FP32 D2Q9 distributions, phi, FP64 water V and E, mask per cell-update


def step_curve(args, config, window=100):
    """ms per step of every ``window``-step block of a fresh run of the 3D
    workload (host wall clock with the device synchronised at each block's
    ends), with the run's heat and water diagnostics at the end."""
    import torch

    from projecticy_amd.iceflow3d import IceFlow3D

    sim = IceFlow3D(config)
    torch.cuda.synchronize()
    curve = []
    for _ in range(args.curve_steps // window):
        start = time.perf_counter()
        sim.step(window)
        torch.cuda.synchronize()
        curve.append(round((time.perf_counter() - start) / window * 1e3, 4))
        if len(curve) % 10 == 0:
            print(f"[bench] curve: {sim.steps} steps, last window {curve[-1]:.3f} ms/step", file=sys.stderr,
                  flush=True)
    out = {"steps": sim.steps, "window": window, "ms_per_step": curve,
           "mean_ms_per_step": round(sum(curve) / len(curve), 4) if curve else None}
    del sim
    torch.cuda.empty_cache()
    return out


def curve_markdown(curve, config, command):
    nx, ny, nz = config.nx, config.ny, config.nz
    lines = [f"# ms per step over a full run: D3Q27 HOME dam break {nx}x{ny}x{nz}, four 16-cell ice cubes", "",
             "Made by (from the repository root, on one MI355X):", "", "```", command, "```", "",
             f"{curve['steps']} coupled steps from initialisation (after the {config.phase_warmup_steps}-step "
             f"phase warm-up), host wall clock over each {curve['window']}-step window with the device "
             f"synchronised at its ends; every {config.thermal.update_interval_lbm_steps}th step adds the heat "
             f"update.  Mean {curve['mean_ms_per_step']:.3f} ms per step.", "",
             "| steps | ms/step | MLUPS |", "|---|---:|---:|"]
    cells = nx * ny * nz
    for k, ms in enumerate(curve["ms_per_step"]):
        lines.append(f"| {k * curve['window'] + 1}-{(k + 1) * curve['window']} | {ms:.3f} | {cells / ms / 1e3:.0f} |")
    return "\n".join(lines) + "\n"


def d2q9_measurement(args):
    """The coupled D2Q9 step on the 1024x2048 falling-ice case (one GPU)."""
    import torch

    from projecticy_amd.iceflow2d import IceFlow2D
    from projecticy_amd.iceflow2d.workloads import scaled_case

    config = scaled_case(seed=args.seed)
    cells = config.nx * config.ny
    t0 = time.perf_counter()
    sim = IceFlow2D(config)
    torch.cuda.synchronize()
    init_s = time.perf_counter() - t0
    sim.step(10)
    torch.cuda.synchronize()
    start = time.perf_counter()
    sim.step(args.d2q9_steps)
    torch.cuda.synchronize()
    seconds = time.perf_counter() - start
    mlups = cells * args.d2q9_steps / seconds / 1e6
    print(f"[bench] D2Q9 {config.nx}x{config.ny}: init {init_s:.1f} s, {args.d2q9_steps} steps in {seconds:.3f} s "
          f"= {mlups:.1f} MLUPS", file=sys.stderr, flush=True)
    result = {
        "workload": f"D2Q9 falling ice {config.nx}x{config.ny}, {config.ice_width}-cell ice at "
                    f"{math.degrees(config.ice_initial_angle):.3f} deg, 90 degC bath, full coupled step",
        "value": round(mlups, 2), "unit": "MLUPS", "steps": args.d2q9_steps,
        "ms_per_step": round(seconds / args.d2q9_steps * 1e3, 4), "dtype": "fp32 populations, fp64 thermal",
        "step_hbm_roofline_frac": round(mlups * 1e6 * D2Q9_STEP_BYTES / (HBM_PEAK_GBS * 1e9), 4),
    }
    counters, stale = measured_counters(COUNTERS_2D, "d2q9")
    fused = (counters or {}).get("kernels", {}).get("k2_collide_push")
    if fused and fused.get("mean_us"):
        seconds = fused["mean_us"] * 1e-6
        traffic = fused.get("read_bytes", 0.0) + fused.get("write_bytes", 0.0)
        result["fused_kernel"] = {
            "kernel": "k2_collide_push", "mean_us": round(fused["mean_us"], 1),
            "bytes_per_cell": D2Q9_FUSED_BYTES,
            "algorithmic_GBs": round(D2Q9_FUSED_BYTES * cells / seconds / 1e9, 1),
            "hbm_GBs_counted": round(traffic / seconds / 1e9, 1), "traffic": round(traffic),
            "valu_busy": None if fused.get("valu_busy") is None else round(fused["valu_busy"], 3),
        }
    else:
        result["fused_kernel"] = {"counters": stale or "no fused-kernel entry"}
    if not args.no_cpu_baseline:
        result["cpu_baseline"] = d2q9_cpu_baseline(config)
    return result


ENSEMBLE_CASE_STEPS = 10000  # steps of one ensemble case


BF16_MFMA_PEAK_TFLOPS = 2500.0  # dense BF16 matrix-core peak of MI355X


def closure_measurement(args):
    """The learned closure's BF16 MFMA kernels on the coarse 128x64x64 grid:
    forward (4 convolutions) and backward (weight gradients of all four,
    data gradients of the last three) of one sample, timed with HIP events."""
    import numpy as np
    import torch

    from projecticy_amd.closure import ClosureNet

    shape = (128, 64, 64)
    cells = shape[0] * shape[1] * shape[2]
    net = ClosureNet(shape, seed=args.seed)
    rng = np.random.default_rng(args.seed)
    feats = torch.from_numpy(rng.normal(size=(cells, 32)).astype(np.float32)).to(torch.bfloat16).cuda()
    feats[:, 8:] = 0
    features = feats.view(torch.int16)
    target = torch.zeros(cells, dtype=torch.float32, device="cuda")
    weight = torch.full((cells,), 1.0 / cells, dtype=torch.float32, device="cuda")
    net.forward(features)
    net.backward(target, weight)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    events = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
    fwd = bwd = 0.0
    for _ in range(args.closure_repeats):
        events[0].record(stream)
        net.forward(features)
        events[1].record(stream)
        net.backward(target, weight)
        events[2].record(stream)
        events[2].synchronize()
        fwd += events[0].elapsed_time(events[1])
        bwd += events[1].elapsed_time(events[2])
    fwd /= args.closure_repeats
    bwd /= args.closure_repeats
    conv = 2.0 * 27 * 32 * 32 * cells  # executed MFMA FLOPs of one 32 -> 32 convolution
    # forward: the first layer as 7 MFMA groups of four taps x 8 channels, two
    # 32 -> 32 layers, the last layer's one 16-channel output tile
    fwd_flops = 2.0 * 7 * 32 * 32 * cells + 2 * conv + conv / 2
    bwd_flops = 7 * conv  # 4 weight + 3 data gradients over 32 padded channels
    algorithmic = 2.0 * 27 * cells * (8 * 32 + 32 * 32 + 32 * 32 + 32 * 1)
    print(f"[bench] closure 128x64x64: forward {fwd:.3f} ms ({fwd_flops / fwd / 1e9:.1f} TFLOP/s), backward "
          f"{bwd:.3f} ms ({bwd_flops / bwd / 1e9:.1f} TFLOP/s)", file=sys.stderr, flush=True)
    result = {
        "workload": "closure CNN, 4 x (3x3x3 conv, 32 channels), BF16 MFMA / FP32 accumulate, 128x64x64 coarse grid",
        "forward_ms": round(fwd, 4), "backward_ms": round(bwd, 4),
        "forward_tflops": round(fwd_flops / fwd / 1e9, 1), "backward_tflops": round(bwd_flops / bwd / 1e9, 1),
        "forward_frac_of_bf16_peak": round(fwd_flops / fwd / 1e9 / BF16_MFMA_PEAK_TFLOPS, 4),
        "forward_algorithmic_tflops": round(algorithmic / fwd / 1e9, 1),
        "note": "executed FLOPs: forward with the 8-channel first layer (four taps per MFMA) and the last layer's one "
                "16-channel tile; backward over 32 padded channels",
    }
    del net
    torch.cuda.empty_cache()
    if args.closure_score_steps > 0:
        result["dam_break"] = closure_dam_break(args)
    return result


CLOSURE_WEIGHTS = ROOT / "projecticy_amd" / "closure" / "weights_128x64x64.npz"


def closure_dam_break(args):
    """The trained closure in the loop of the halved dam break (128x64x64,
    a geometry outside its training pairs) against the same tank at twice
    the resolution, over ``--closure-score-steps`` coarse steps."""
    from projecticy_amd.closure import ClosureNet
    from projecticy_amd.closure.experiment import dam_break_score, load_weights

    if not CLOSURE_WEIGHTS.exists():
        return {"skipped": f"no trained weights at {CLOSURE_WEIGHTS.relative_to(ROOT)}"}
    net = ClosureNet((128, 64, 64), seed=args.seed)
    load_weights(net, CLOSURE_WEIGHTS)
    t0 = time.perf_counter()
    out = dam_break_score(net, seed=args.seed, steps=args.closure_score_steps)
    out["seconds"] = round(time.perf_counter() - t0, 1)
    out["weights"] = str(CLOSURE_WEIGHTS.relative_to(ROOT))
    # The melted masses and centre trajectories of dam_break_score are for
    # plots; in the one line of results they were most of 9 KB.
    del out["melted_kg"], out["centres_m"]
    print(f"[bench] closure dam break {out['coarse_steps']} coarse steps in {out['seconds']} s: final melt error "
          f"plain {out['plain']['final_melt_error']:.3f}, closure {out['closure']['final_melt_error']:.3f}; "
          f"max centroid error plain {out['plain']['max_centroid_error_m']:.2e} m, closure "
          f"{out['closure']['max_centroid_error_m']:.2e} m", file=sys.stderr, flush=True)
    return out


ENSEMBLE_STORAGE = ("fp16-momentum-sr", "fp32", "fp16-rel-sr")
HEADLINE_STORAGE = "fp16-momentum-sr"  # FP16 populations (momentum), FP32 arithmetic


def ensemble_measurement(args):
    """64 uneven D2Q9 cases stepped as one batch (one launch per kernel for
    all cases), for each population storage; cases/hour against the same
    cases run one at a time with FP32 populations; and, from the fine-solver
    gate, how many of those cases melt within 1% of the fine plain solver."""
    import torch

    from projecticy_amd.iceflow2d import IceFlow2D
    from projecticy_amd.iceflow2d.ensemble import IceFlowEnsemble2D
    from projecticy_amd.iceflow2d.workloads import ensemble_cases, ensemble_draws

    configs = ensemble_cases(args.ensemble_cases, seed=args.seed)
    draws = ensemble_draws(args.ensemble_cases, seed=args.seed)
    storages = {}
    cells = 0
    for storage in ENSEMBLE_STORAGE:
        t0 = time.perf_counter()
        ensemble = IceFlowEnsemble2D(configs, population_storage=storage)
        init_s = time.perf_counter() - t0
        tuning = ensemble.autotune()
        ensemble.step(8)
        torch.cuda.synchronize()
        start = time.perf_counter()
        ensemble.step(args.ensemble_steps)
        torch.cuda.synchronize()
        seconds = time.perf_counter() - start
        cells = ensemble.cells
        per_step = seconds / args.ensemble_steps
        storages[storage] = {
            "cases_per_hour": round(len(configs) * 3600.0 / (per_step * ENSEMBLE_CASE_STEPS), 2),
            "ms_per_step": round(per_step * 1e3, 4),
            "mlups": round(cells * args.ensemble_steps / seconds / 1e6, 2),
            "threads": list(ensemble.threads),
            "autotune_ms_per_step": {f"{c}/{s}": round(t * 1e3, 3) for (c, s), t in tuning.items()},
        }
        print(f"[bench] ensemble {storage}: {len(configs)} cases, {cells / 1e6:.2f} M cells, init {init_s:.1f} s, "
              f"{args.ensemble_steps} steps in {seconds:.3f} s, {storages[storage]['cases_per_hour']:.1f} cases/h",
              file=sys.stderr, flush=True)
        del ensemble
        torch.cuda.empty_cache()
    # plain form: each case alone, FP32 populations, one width at a time
    plain_step = {}
    for config in configs:
        if config.nx in plain_step:
            continue
        sim = IceFlow2D(config)
        sim.step(8)
        torch.cuda.synchronize()
        begin = time.perf_counter()
        sim.step(16)
        torch.cuda.synchronize()
        plain_step[config.nx] = (time.perf_counter() - begin) / 16
        del sim
    plain_cases_hour = len(configs) * 3600.0 / sum(plain_step[c.nx] * ENSEMBLE_CASE_STEPS for c in configs)
    result = {
        "workload": f"{len(configs)} D2Q9 falling-ice cases, widths 64-512 (height 2x), seed {args.seed}, "
                    f"{ENSEMBLE_CASE_STEPS} steps per case, batched launches",
        "unit": "cases/hour", "cells": cells, "steps_timed": args.ensemble_steps,
        "plain_fp32_cases_per_hour": round(plain_cases_hour, 2),
        "storage": storages,
    }
    if args.ensemble_gate_steps > 0:
        gate = fine_solver_gate(configs, draws, args.ensemble_gate_steps)
        result["fine_solver_gate"] = gate
        for storage, entry in storages.items():
            passed = gate["within_1pct_by_width"][storage]
            valid = sum(1 for c in configs if passed[str(c.nx)])
            entry["cases_within_1pct"] = valid
            entry["cases_per_hour_within_1pct"] = round(entry["cases_per_hour"] * valid / len(configs), 2)
            # the same count with the melt difference taken as a fraction of the initial ice mass
            passed_ice = gate["within_1pct_of_ice_by_width"][storage]
            entry["cases_within_1pct_of_ice_mass"] = sum(1 for c in configs if passed_ice[str(c.nx)])
    headline = storages[HEADLINE_STORAGE]
    result["value"] = headline.get("cases_per_hour_within_1pct")
    result["storage_at_value"] = HEADLINE_STORAGE
    result["speedup_vs_plain"] = round(headline["cases_per_hour"] / plain_cases_hour, 3)
    print(f"[bench] ensemble ({HEADLINE_STORAGE}): {headline['cases_per_hour']} cases/h, "
          f"{headline.get('cases_within_1pct')} of {len(configs)} cases within 1% of the fine solver -> "
          f"{result['value']} cases/h; plain FP32 {plain_cases_hour:.1f} cases/h", file=sys.stderr, flush=True)
    return result


def fine_solver_gate(configs, draws, steps):
    """Melted mass after ``steps`` coarse steps, per storage, of one case of
    each width (the first drawn), against the fine plain solver: the same case
    on a twice finer grid (FP32 populations) over the same physical time
    (2 x steps).  A width passes when its case's melted mass is within 1% of
    the fine solver's; the cases/hour count only the cases of passing widths
    (the per-width case stands for the other cases of its width)."""
    import torch

    from projecticy_amd.iceflow2d.ensemble import IceFlowEnsemble2D
    from projecticy_amd.iceflow2d.workloads import refined_case

    picked, widths = [], set()
    for config, draw in zip(configs, draws):
        if config.nx not in widths:
            widths.add(config.nx)
            picked.append((config, draw))
    t0 = time.perf_counter()
    fine = IceFlowEnsemble2D([refined_case(d) for _, d in picked], population_storage="fp32")
    fine.autotune()
    fine.step(2 * steps)
    fine_melt = [t.melted_mass_kg_m for t in fine.totals()]
    fine_ice0 = [t.initial_body_mass_kg_m for t in fine.totals()]
    del fine
    torch.cuda.empty_cache()
    print(f"[bench] fine solver: {len(picked)} cases x {2 * steps} steps in {time.perf_counter() - t0:.1f} s",
          file=sys.stderr, flush=True)
    melted, errors, passed, ice_errors, passed_ice = {}, {}, {}, {}, {}
    for storage in ENSEMBLE_STORAGE:
        batch = IceFlowEnsemble2D([c for c, _ in picked], population_storage=storage)
        batch.autotune()
        batch.step(steps)
        totals = batch.totals()
        del batch
        torch.cuda.empty_cache()
        melted[storage] = [t.melted_mass_kg_m for t in totals]
        errors[storage] = [abs(a - b) / b if b > 0.0 else None for a, b in zip(melted[storage], fine_melt)]
        # the same difference as a fraction of the initial ice mass
        ice_errors[storage] = [abs(a - b) / m for a, b, m in zip(melted[storage], fine_melt, fine_ice0)]
        passed[storage] = {str(c.nx): e is not None and e <= 0.01 for (c, _), e in zip(picked, errors[storage])}
        passed_ice[storage] = {str(c.nx): e <= 0.01 for (c, _), e in zip(picked, ice_errors[storage])}
    worst = {k: max(e for e in v if e is not None) for k, v in errors.items()}
    print(f"[bench] fine-solver gate: {len(picked)} widths x {steps} steps, melted-mass error vs fine "
          + ", ".join(f"{k} max {v:.3e}" for k, v in worst.items()), file=sys.stderr, flush=True)
    short = lambda values: [None if v is None else float(f"{v:.4g}") for v in values]  # noqa: E731
    return {
        "steps": steps, "fine_steps": 2 * steps, "widths": [c.nx for c, _ in picked],
        "melted_kg_m_fine": short(fine_melt),
        "melted_mass_relative_error": {k: short(v) for k, v in errors.items()},
        "error_fraction_of_initial_ice": {k: short(v) for k, v in ice_errors.items()},
        "max_relative_error": {k: float(f"{v:.4g}") for k, v in worst.items()},
        "within_1pct_by_width": passed, "within_1pct_of_ice_by_width": passed_ice,
        "reference": "the same case on a twice finer grid, FP32 populations, over the same physical time",
    }


def host_cpu():
    """(threads the OpenMP oracle runs on, CPU model name)."""
    threads = int(os.environ.get("OMP_NUM_THREADS") or os.cpu_count() or 1)
    model = "unknown"
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return threads, model


D2Q9_CPU_STEPS = 8
D2Q9_CPU_WARMUP = 40  # a shortened phase warm-up (the full 500 steps take minutes on the CPU)


def d2q9_cpu_baseline(config):
    """The FP64 C oracle (OpenMP over the host's cores) on a window of the
    same 1024x2048 case: 8 coupled steps (one slow thermal update) after
    initialisation with a 40-step phase warm-up and one untimed step."""
    from dataclasses import replace

    from oracle.iceflow2d_oracle import Oracle2D, build_oracle2d

    build_oracle2d()
    ref = Oracle2D(replace(config, phase_warmup_steps=D2Q9_CPU_WARMUP))
    ref.step(1)
    start = time.perf_counter()
    ref.step(D2Q9_CPU_STEPS)
    seconds = time.perf_counter() - start
    threads, model = host_cpu()
    return {"value": config.nx * config.ny * D2Q9_CPU_STEPS / seconds / 1e6, "unit": "MLUPS", "cores": threads,
            "kind": "port", "cpu": model,
            "sample": f"{D2Q9_CPU_STEPS} coupled steps (one slow thermal update) of the same {config.nx}x{config.ny} "
                      f"case after initialisation with a {D2Q9_CPU_WARMUP}-step phase warm-up and one untimed step, {seconds:.2f} s, FP64 "
                      f"C oracle, OpenMP on {threads} threads"}


CPU_STEPS = 8


def cpu_baseline(config):
    """The FP64 C oracle (OpenMP over the host's cores) on a window of the
    same workload: 8 coupled steps, the eighth with the conduction and melt
    update, after initialisation without the phase warm-up."""
    from dataclasses import replace

    from oracle.iceflow3d_oracle import Oracle3D, build_oracle

    build_oracle()
    ref = Oracle3D(replace(config, phase_warmup_steps=0))
    start = time.perf_counter()
    ref.step(CPU_STEPS)
    seconds = time.perf_counter() - start
    cells = config.nx * config.ny * config.nz
    threads, model = host_cpu()
    return {
        "value": cells * CPU_STEPS / seconds / 1e6,
        "unit": "MLUPS",
        "cores": threads,
        "kind": "port",
        "cpu": model,
        "sample": f"{CPU_STEPS} coupled steps (the eighth with conduction and melting) of the same "
                  f"{config.nx}x{config.ny}x{config.nz} workload after initialisation without phase warm-up, "
                  f"{seconds:.2f} s, FP64 C oracle, OpenMP on {threads} threads",
    }


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {args.gpus}); the multi-GPU decomposition "
              "is a design (slab halos over RCCL) with no runnable path in this build", file=sys.stderr)
        sys.exit(2)
    import torch

    from projecticy_amd.iceflow3d import IceFlow3D
    from projecticy_amd.iceflow3d.workloads import dam_break_four_ice

    nx, ny, nz = args.size
    config = dam_break_four_ice(nx, ny, nz, seed=args.seed)
    cells = nx * ny * nz
    t0 = time.perf_counter()
    sim = IceFlow3D(config)
    torch.cuda.synchronize()
    init_s = time.perf_counter() - t0
    print(f"[bench] initialised {nx}x{ny}x{nz} in {init_s:.1f} s", file=sys.stderr, flush=True)
    sim.step(args.warmup)
    torch.cuda.synchronize()
    start = time.perf_counter()
    sim.step(args.steps)
    torch.cuda.synchronize()
    seconds = time.perf_counter() - start
    mlups = cells * args.steps / seconds / 1e6
    print(f"[bench] {args.steps} steps in {seconds:.3f} s = {mlups:.1f} MLUPS", file=sys.stderr, flush=True)

    sim.attach_profiler()
    sim.step(args.profile_steps)
    torch.cuda.synchronize()
    totals = sim.profile_totals()
    sim.detach_profiler()
    counters, stale = measured_counters()
    counted = counters["groups"] if counters else {}
    groups = {}
    for name, (ms, count) in totals.items():
        mean_ms = ms / max(count, 1)
        gbs = KERNEL_BYTES[name] * cells / (mean_ms * 1e-3) / 1e9 if mean_ms > 0 else 0.0
        groups[name] = {"mean_ms": round(mean_ms, 5), "algorithmic_GBs": round(gbs, 1)}
        if name in counted and mean_ms > 0:
            groups[name]["hbm_GBs_counted"] = round(counted[name]["traffic_bytes"] / (mean_ms * 1e-3) / 1e9, 1)
            if counted[name].get("valu_busy") is not None:
                groups[name]["valu_busy_counted"] = round(counted[name]["valu_busy"], 3)
    dominant = max(groups, key=lambda k: groups[k]["mean_ms"])
    achieved = groups[dominant]["algorithmic_GBs"]
    roofline = {
        "bound": "hbm",
        "achieved": achieved,
        "peak": HBM_PEAK_GBS,
        "unit": "GB/s",
        "frac": round(achieved / HBM_PEAK_GBS, 4),
        "traffic": round(counted[dominant]["traffic_bytes"]) if dominant in counted else None,
        "kernel": dominant,
        "bytes_per_cell": KERNEL_BYTES[dominant],
        "cells_per_launch": cells,
        "valu_busy": groups[dominant].get("valu_busy_counted"),
        "counters": "current" if counters else stale,
    }
    result = {
        "metric": "D3Q27 MLUPS + % HBM roofline; ensemble cases/hour at <=1% melt-mass error",
        "value": round(mlups, 2),
        "unit": "MLUPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(seconds / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic",
        "config": {
            "workload": f"D3Q27 HOME dam break {nx}x{ny}x{nz}, four seeded 16-cell ice cubes, full coupled step",
            "grid": [nx, ny, nz],
            "seed": args.seed,
            "bodies": len(config.bodies),
            "phase_warmup_steps": config.phase_warmup_steps,
            "thermal_interval": config.thermal.update_interval_lbm_steps,
        },
        "step_hbm_roofline_frac": round(mlups * 1e6 * STEP_BYTES / (HBM_PEAK_GBS * 1e9), 4),
        "kernel_groups": groups,
        "roofline": roofline,
        "cpu_baseline": None if args.no_cpu_baseline else cpu_baseline(config),
    }
    del sim
    torch.cuda.empty_cache()
    if args.curve_steps > 0:
        result["curve"] = step_curve(args, config)
        if args.curve_md is not None:
            args.curve_md.write_text(curve_markdown(result["curve"], config, "python3 " + " ".join(sys.argv)))
    if args.d2q9_steps > 0:
        result["d2q9"] = d2q9_measurement(args)
        torch.cuda.empty_cache()
    if args.ensemble_steps > 0:
        result["ensemble"] = ensemble_measurement(args)
    if args.closure_repeats > 0:
        result["closure"] = closure_measurement(args)
    if args.copy_probe_mib > 0:
        src = torch.ones(args.copy_probe_mib * (1 << 18), dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(5):
            torch.mul(src, 1.0, out=dst)
        torch.cuda.synchronize()
        del src, dst
    # measured last, so that a counter run's step window (which ends at the
    # copy probe above) holds no copy of this size
    copy_gbs = copy_bandwidth()
    roofline["copy_GBs_measured"] = round(copy_gbs, 1)
    roofline["frac_of_copy"] = round(achieved / copy_gbs, 4)
    result["step_frac_of_copy"] = round(mlups * 1e6 * STEP_BYTES / (copy_gbs * 1e9), 4)
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
