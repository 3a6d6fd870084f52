"""Turn rocprofv3 runs of ``bench.py`` into the counter summary it reports.

Three counter passes and one kernel trace of the same short bench command
(each pass its own process, as rocprofv3 collects one counter group per run).
For the 3D dam break (``--workload dam_break``, the default):

    CMD="python3 bench.py --steps 6 --warmup 2 --profile-steps 0 --d2q9-steps 0 \\
         --ensemble-steps 0 --closure-repeats 0 --no-cpu-baseline --copy-probe-mib 1024"
    rocprofv3 --kernel-trace --stats --output-format csv -d gpurun_out/prof_trace -o run -- $CMD
    rocprofv3 --pmc FETCH_SIZE --output-format csv -d gpurun_out/prof_fetch -o run -- $CMD
    rocprofv3 --pmc WRITE_SIZE --output-format csv -d gpurun_out/prof_write -o run -- $CMD
    rocprofv3 --pmc SQ_INSTS_VALU SQ_ACTIVE_INST_VALU GRBM_GUI_ACTIVE --output-format csv \\
         -d gpurun_out/prof_valu -o run -- $CMD
    python3 profile_counters.py gpurun_out/prof_trace gpurun_out/prof_fetch gpurun_out/prof_write \\
         gpurun_out/prof_valu --out profiles/counters_dam_break_256x128x128

For the D2Q9 1024x2048 case (``--workload d2q9``) the bench command runs
two 3D steps and the 2D measurement, and the window starts at the first
2D fused collide-and-push pass:

    CMD="python3 bench.py --steps 2 --warmup 0 --profile-steps 0 --d2q9-steps 100 \\
         --ensemble-steps 0 --closure-repeats 0 --no-cpu-baseline --copy-probe-mib 1024"
    ... the same four rocprofv3 runs into gpurun_out/prof2d_{trace,fetch,write,valu} ...
    python3 profile_counters.py --workload d2q9 gpurun_out/prof2d_trace gpurun_out/prof2d_fetch \\
         gpurun_out/prof2d_write gpurun_out/prof2d_valu --out profiles/counters_d2q9_falling_ice_1024x2048

The script keeps the dispatches of the timed step (from the workload's
first flow kernel on, before the copy probe), averages each counter per
kernel, scales FETCH_SIZE and WRITE_SIZE (KiB per dispatch) to bytes by what
they read for the copy probe (``--copy-probe-mib`` of FP32 read and written
once), and writes ``<out>.json`` (read by bench.py, stamped with the hash of
the kernel sources it was measured on) and ``<out>.md``.
"""

import argparse
import csv
import hashlib
import json
import re
import sys
from collections import defaultdict
from pathlib import Path

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "projecticy_amd" / "csrc"
SIMDS = 256 * 4  # MI355X: 256 CUs of four SIMDs
XCDS = 8  # GRBM_GUI_ACTIVE is reported summed over the eight XCDs

# Per workload: the step's first kernel, the cells of one step, and the
# bench's kernel groups (bench.py KERNEL_BYTES for the 3D flow step).
WORKLOADS = {
    "dam_break": {
        "title": "D3Q27 HOME dam break 256x128x128", "cells": 256 * 128 * 128, "first": "k_stream_rows",
        "groups": {
            "phase_collide": ("k_collide_phase",),
            "forces": ("k_forces_rows", "k_forces_general", "k_classify", "k_scatter_flags"),
            "home_collide_stream": ("k_stream_rows", "k_stream_boundary", "k_finish_loads"),
            "phase_recover": ("k_recover_phase", "k_fold_recovery"),
            "gradients": ("k_gradients_tiled", "k_gradients_general_list"),
        },
    },
    "d2q9": {
        "title": "D2Q9 falling ice 1024x2048", "cells": 1024 * 2048, "first": "k2_collide_push",
        "groups": {"collide_stream": ("k2_collide_push",)},
    },
}
PROBE_KERNEL = "MulFunctor"


# The kernel sources each workload's counters describe.
SOURCES = {
    "dam_break": ("csrc/icy3d_*.hip", "csrc/icy3d_device.h", "../include/icy3d.h"),
    "d2q9": ("csrc/icy2d.hip", "../include/icy2d.h"),
}


def source_hash(workload="dam_break"):
    """SHA-256 over the HIP sources and headers of the workload's kernels and
    the compiler flags they are built with (the include path left out)."""
    from projecticy_amd.build import HIP_FLAGS

    base = ROOT / "projecticy_amd"
    paths = sorted({p.resolve() for pattern in SOURCES[workload] for p in base.glob(pattern)})
    h = hashlib.sha256()
    for path in paths:
        h.update(path.name.encode())
        h.update(path.read_bytes())
    h.update(" ".join(f for f in HIP_FLAGS if f != "-I" and not f.startswith("/")).encode())
    return h.hexdigest()[:16]


def short_name(kernel):
    """``void icy::k_stream_boundary<true>(icy3d_grid) [clone .kd]`` or
    ``(anonymous namespace)::k_finish_sum(float const*, int, float*)`` ->
    the bare function name; the 2D launch wrappers ``one_case<T, &F, ...>``
    and ``many_cases<T, &F, ...>`` -> F."""
    name = kernel.replace("(anonymous namespace)::", "")
    mangled = re.search(r"(?:one_case|many_cases)ILi\d+ETnDaXadL_ZNS_(\d+)", name)
    if mangled:  # _ZN4icy28one_caseILi256ETnDaXadL_ZNS_9k2_streamE...: length-prefixed name
        return name[mangled.end():mangled.end() + int(mangled.group(1))]
    wrapped = re.search(r"(?:one_case|many_cases)<\s*\d+\s*,\s*\(?&?\(?([\w:]+)", name)
    if wrapped:
        return wrapped.group(1).split("::")[-1]
    name = name.split("(")[0].strip()
    name = name.split()[-1] if name else kernel
    return name.split("<")[0].split("::")[-1]


def _csv_rows(folder, suffix):
    files = sorted(Path(folder).rglob(f"*{suffix}"))
    if not files:
        raise SystemExit(f"no *{suffix} under {folder}")
    for path in files:
        with path.open(newline="") as handle:
            yield from csv.DictReader(handle)


def counter_dispatches(folder):
    """{dispatch id: (kernel, {counter: value})} of one --pmc run."""
    out = {}
    for row in _csv_rows(folder, "counter_collection.csv"):
        key = int(row["Dispatch_Id"])
        kernel, values = out.setdefault(key, (row["Kernel_Name"], {}))
        values[row["Counter_Name"]] = values.get(row["Counter_Name"], 0.0) + float(row["Counter_Value"])
    return out


def trace_dispatches(folder):
    """{dispatch id: (kernel, start ns, end ns)} of a --kernel-trace run."""
    out = {}
    for row in _csv_rows(folder, "kernel_trace.csv"):
        out[int(row["Dispatch_Id"])] = (row["Kernel_Name"], int(row["Start_Timestamp"]), int(row["End_Timestamp"]))
    return out


def step_spans(trace, window, first):
    """Wall time of the traced steps: the span from one fused collide-stream's
    start to the next one's and the kernel time inside it, as medians over
    the steps (every eighth step adds the heat update)."""
    starts = [trace[i][1] for i in window if short_name(trace[i][0]) == first]
    spans, busy = [], []
    for a, b in zip(starts, starts[1:]):
        spans.append(b - a)
        busy.append(sum(trace[i][2] - trace[i][1] for i in window if a <= trace[i][1] < b))
    idle = sorted(s - k for s, k in zip(spans, busy))
    median = lambda v: sorted(v)[len(v) // 2] / 1e3  # noqa: E731
    return {"steps": len(spans), "median_step_us": median(spans), "median_kernel_us": median(busy),
            "median_idle_us": median(idle)}


def step_window(dispatches, first_kernel):
    """Dispatch ids of the timed steps: from the first ``first_kernel``
    dispatch up to (not including) the first copy-probe dispatch."""
    ids = sorted(dispatches)
    first = next(i for i in ids if short_name(dispatches[i][0]) == first_kernel)
    last = next((i for i in ids if i > first and PROBE_KERNEL in dispatches[i][0]), ids[-1] + 1)
    return [i for i in ids if first <= i < last]


def probe_values(dispatches, counter):
    values = [v[counter] for k, v in dispatches.values() if PROBE_KERNEL in k and counter in v]
    if not values:
        raise SystemExit(f"no copy-probe dispatch with {counter}")
    return sum(values) / len(values)


def per_kernel(dispatches, window, counters):
    sums, counts = defaultdict(lambda: defaultdict(float)), defaultdict(int)
    for i in window:
        kernel, values = dispatches[i]
        name = short_name(kernel)
        counts[name] += 1
        for c in counters:
            sums[name][c] += values.get(c, 0.0)
    return {name: {c: sums[name][c] / counts[name] for c in counters} | {"dispatches": counts[name]}
            for name in counts}


def summarise(trace_dir, fetch_dir, write_dir, valu_dir, probe_mib, workload="dam_break"):
    spec = WORKLOADS[workload]
    first = spec["first"]
    probe_kib = probe_mib * 1024.0
    fetch, write, valu = (counter_dispatches(d) for d in (fetch_dir, write_dir, valu_dir))
    read_scale = probe_kib / probe_values(fetch, "FETCH_SIZE")
    write_scale = probe_kib / probe_values(write, "WRITE_SIZE")
    kernels = defaultdict(dict)
    for name, v in per_kernel(fetch, step_window(fetch, first), ["FETCH_SIZE"]).items():
        kernels[name].update(read_bytes=v["FETCH_SIZE"] * 1024.0 * read_scale, dispatches=v["dispatches"])
    for name, v in per_kernel(write, step_window(write, first), ["WRITE_SIZE"]).items():
        kernels[name]["write_bytes"] = v["WRITE_SIZE"] * 1024.0 * write_scale
    names = ["SQ_INSTS_VALU", "SQ_ACTIVE_INST_VALU", "GRBM_GUI_ACTIVE"]
    for name, v in per_kernel(valu, step_window(valu, first), names).items():
        kernels[name]["valu_insts"] = v["SQ_INSTS_VALU"]
        cycles = v["GRBM_GUI_ACTIVE"] / XCDS  # GPU-busy cycles of the dispatch
        # rocprof's derived VALUBusy: each VALU instruction of a wave64 occupies
        # its SIMD for 4 cycles; the fraction of all SIMDs' cycles so spent
        kernels[name]["valu_busy"] = 4.0 * v["SQ_ACTIVE_INST_VALU"] / SIMDS / cycles if cycles else None
    spans = None
    if trace_dir:
        trace = trace_dispatches(trace_dir)
        window = step_window(trace, first)
        durations = defaultdict(list)
        for i in window:
            durations[short_name(trace[i][0])].append(trace[i][2] - trace[i][1])
        for name, values in durations.items():
            kernels[name]["mean_us"] = sum(values) / len(values) / 1e3
        spans = step_spans(trace, window, first)
    groups = {}
    for group, members in spec["groups"].items():
        present = [kernels[m] for m in members if m in kernels]
        steps = max((k.get("dispatches", 0) for k in present), default=0)
        if not present or not steps:
            continue
        # bytes per step of the group: each member's mean times its dispatches per step
        per_step = lambda key: sum(k.get(key, 0.0) * k.get("dispatches", 0) for k in present) / steps  # noqa: E731
        groups[group] = {"traffic_bytes": per_step("read_bytes") + per_step("write_bytes"),
                         "read_bytes": per_step("read_bytes"), "write_bytes": per_step("write_bytes")}
        main = kernels.get(members[0], {})
        if main.get("valu_busy") is not None:
            groups[group]["valu_busy"] = main["valu_busy"]
    return {
        "source_sha": source_hash(workload),
        "calibration": {"probe_mib": probe_mib, "read_bytes_per_fetch_kib": 1024.0 * read_scale,
                        "write_bytes_per_write_kib": 1024.0 * write_scale},
        "kernels": {k: dict(v) for k, v in sorted(kernels.items())},
        "groups": groups,
        "trace": spans,
        "workload": workload,
        "cells": spec["cells"],
    }


def markdown(summary, command):
    cal = summary["calibration"]
    first = WORKLOADS[summary["workload"]]["first"]
    lines = [
        f"# HBM and VALU counters: {WORKLOADS[summary['workload']]['title']} ({summary['cells']:,} cells)", "",
        f"Kernel sources: `{summary['source_sha']}` (SHA-256 prefix over "
        f"{', '.join('`' + p.replace('../', '') + '`' for p in SOURCES[summary['workload']])} under "
        "`projecticy_amd/` and the hipcc flags of `projecticy_amd/build.py`; bench.py reports these figures only "
        "while the sources and flags hash to it).", "",
        "Made by (from the repository root, on one MI355X; `TMPDIR=/tmp`):", "", "```", command, "```", "",
        f"**Calibration.** The copy probe reads and writes {cal['probe_mib']} MiB of FP32 per dispatch; "
        f"one KiB of FETCH_SIZE stands for {cal['read_bytes_per_fetch_kib']:.0f} B read and one KiB of "
        f"WRITE_SIZE for {cal['write_bytes_per_write_kib']:.0f} B written.", "",
    ]
    spans = summary.get("trace")
    if spans:
        lines += [
            f"**Steps.** {spans['steps']} traced steps (medians): {spans['median_step_us']:.0f} us from one "
            f"`{first}` to the next, {spans['median_kernel_us']:.0f} us of kernel time in it and "
            f"{spans['median_idle_us']:.0f} us with no kernel running (launch gaps and the host's decisions "
            "and control reads).", ""]
    lines += [
        f"Per-dispatch means over the timed steps (from the first `{first}` to the copy probe):", "",
        "| kernel | dispatches | read MB | written MB | B/cell | VALU insts (M) | VALUBusy | mean us |",
        "|---|---:|---:|---:|---:|---:|---:|---:|",
    ]
    cells = summary["cells"]
    for name, k in sorted(summary["kernels"].items(), key=lambda kv: -kv[1].get("mean_us", 0.0)):
        if not (name.startswith("k_") or name.startswith("k2_")):
            continue
        rb, wb = k.get("read_bytes", 0.0), k.get("write_bytes", 0.0)
        busy = k.get("valu_busy")
        lines.append(f"| `{name}` | {k.get('dispatches', 0)} | {rb / 1e6:.1f} | {wb / 1e6:.1f} | "
                     f"{(rb + wb) / cells:.1f} | {k.get('valu_insts', 0.0) / 1e6:.2f} | "
                     f"{'' if busy is None else f'{busy:.3f}'} | {k.get('mean_us', 0.0):.1f} |")
    lines += ["", "Per bench kernel group (bytes per step):", "", "| group | traffic MB | B/cell | VALUBusy |",
              "|---|---:|---:|---:|"]
    for name, g in summary["groups"].items():
        busy = g.get("valu_busy")
        lines.append(f"| {name} | {g['traffic_bytes'] / 1e6:.1f} | {g['traffic_bytes'] / cells:.1f} | "
                     f"{'' if busy is None else f'{busy:.3f}'} |")
    return "\n".join(lines) + "\n"


def main(argv=None):
    p = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    p.add_argument("trace", help="rocprofv3 --kernel-trace output folder ('-' for none)")
    p.add_argument("fetch")
    p.add_argument("write")
    p.add_argument("valu")
    p.add_argument("--probe-mib", type=int, default=1024)
    p.add_argument("--workload", choices=sorted(WORKLOADS), default="dam_break")
    p.add_argument("--out", type=Path, required=True, help="output path without suffix")
    p.add_argument("--command", default="(see profile_counters.py)", help="the command recorded in the summary")
    args = p.parse_args(argv)
    summary = summarise(None if args.trace == "-" else args.trace, args.fetch, args.write, args.valu, args.probe_mib,
                        args.workload)
    args.out.with_suffix(".json").write_text(json.dumps(summary, indent=1) + "\n")
    args.out.with_suffix(".md").write_text(markdown(summary, args.command))
    print(json.dumps(summary["groups"], indent=1))


if __name__ == "__main__":
    sys.exit(main())
