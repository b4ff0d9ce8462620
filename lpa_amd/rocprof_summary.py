"""Text summaries of rocprofv3 output for the benchmark's headline phase.

The benchmark's profiled command (bench.py --headline-only ...) builds the
graph, lays it out (with --no-learned the degree schedule; otherwise the
judged learned schedule), the last k_relayout dispatch, and then runs
warm-up and timed iterations, eager at the end.  A step ends with one
k_publish per stream that it used.  A timed iteration is two steps: the step as
it runs, with small bins merged (k_bins) and heavy sets on other streams, and
the same step with a launch per bin on one stream.  The kernel table is of the
first kind, times and traffic per family are of the second, whose launches
belong to one family each.
The copy kernel of the calibration (bench.py --copy-calibration:
k_calibration_copy over 256 MiB) gives the factor between FETCH_SIZE /
WRITE_SIZE readings and bytes actually moved.

Usage:
  python -m lpa_amd.rocprof_summary --trace DIR [--fetch DIR --write DIR]
      --steps S [--pmc-steps S] --command "..."
      --workload W --K K --out PREFIX
writes PREFIX_kernels.txt and PREFIX_traffic.json.
"""
import argparse
import collections
import csv
import json
import os
import re

COPY_BYTES = 256 * 1024 * 1024


def family(name):
    """kernel family (bin kind) of a dispatch, from its demangled name"""
    m = re.search(r"lpa::(k_\w+)(<[^(]*>)?", name)
    if not m:
        return "other"
    k, targs = m.group(1), (m.group(2) or "")
    args = [a.strip() for a in targs.strip("<>").split(",")] if targs else []
    if k == "k_lane":
        return "lane"
    if k == "k_group":
        return "block" if args and args[0] == "256" else "wave"
    if k in ("k_heavy_decode", "k_heavy_clear", "k_heavy_finish", "k_heavy_local"):
        return "cms" if args and args[0] == "1" else "global"
    if k == "k_heavy_chunks":
        return "global" if args and args[0] == "0" else "cms"
    if k == "k_calibration_copy":
        return "copy"
    if k == "k_bins":
        return "bins"
    if k == "k_decode_bins":
        return "cglp-decode"
    if k == "k_publish":
        return "step"
    return "other"


def _rows(path):
    with open(path, newline="") as f:
        return list(csv.DictReader(f))


def _headline(rows, steps):
    """(rows of the steps as run, rows of the steps launched bin by bin) of the
    last `steps` timed iterations, and the calibration copies"""
    rows = sorted(rows, key=lambda r: int(r["Dispatch_Id"]))
    last = max((i for i, r in enumerate(rows) if "k_relayout" in r["Kernel_Name"]), default=-1)
    rows = rows[last + 1:]
    copies = [r for r in rows if family(r["Kernel_Name"]) == "copy"]
    done, ended = [[]], False
    for r in rows:
        f = family(r["Kernel_Name"])
        if f in ("copy", "other"):
            continue
        if ended and f != "step":
            done.append([])
        done[-1].append(r)
        ended = f == "step"
    if not ended:
        done.pop()   # cut off within a step
    if len(done) < 2 * steps:
        raise SystemExit(f"{len(done)} steps after the last layout: {steps} timed iterations make {2 * steps}")
    done = done[-2 * steps:]
    run, alone = sum(done[::2], []), sum(done[1::2], [])
    if any(family(r["Kernel_Name"]) == "bins" for r in alone):
        raise SystemExit("merged bins in a step that launches them one by one: the last steps are not timed eager ones")
    return run, alone, copies


def trace_summary(trace_dir, steps):
    run, alone, _ = _headline(_rows(os.path.join(trace_dir, "run_kernel_trace.csv")), steps)
    us = lambda r: (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3
    per = collections.defaultdict(lambda: [0, 0.0])
    for r in run:
        k = r["Kernel_Name"]
        per[k][0] += 1
        per[k][1] += us(r)
    fam = collections.defaultdict(float)
    for r in alone:
        fam[family(r["Kernel_Name"])] += us(r) / steps / 1e3   # ms per iteration
    return per, fam


def counter_summary(dirname, counter, steps):
    rows = [r for r in _rows(os.path.join(dirname, "run_counter_collection.csv")) if r["Counter_Name"] == counter]
    _, alone, copies = _headline(rows, steps)
    value = lambda r: float(r["Counter_Value"]) * 1024.0   # KiB -> bytes
    fam = collections.defaultdict(float)
    for r in alone:
        fam[family(r["Kernel_Name"])] += value(r) / steps
    return fam, [value(r) for r in copies]


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--trace", required=True)
    ap.add_argument("--fetch")
    ap.add_argument("--write")
    ap.add_argument("--iters", type=int, help="warmup + timed iterations of the trace run (named in the summary)")
    ap.add_argument("--steps", type=int, required=True, help="timed iterations of the trace run (summarised)")
    ap.add_argument("--pmc-iters", type=int, help="warmup + timed iterations of the counter runs")
    ap.add_argument("--pmc-steps", type=int, help="timed iterations of the counter runs")
    ap.add_argument("--command", required=True, help="profiled command lines, ';'-separated")
    ap.add_argument("--workload", required=True)
    ap.add_argument("--K", type=int, required=True)
    ap.add_argument("--out", required=True)
    a = ap.parse_args()
    per, fam = trace_summary(a.trace, a.steps)
    lines = [f"rocprofv3 kernel trace, headline phase of {a.workload} K={a.K}: the {a.steps} timed iterations "
             f"{f'(of {a.iters}) ' if a.iters else ''}after the last layout build", "commands:"]
    lines += [f"  {c.strip()}" for c in a.command.split(";") if c.strip()]
    lines.append("")
    lines.append(f"{'kernel':78s} {'calls':>6s} {'avg_us':>9s} {'us/iter':>9s} family")
    for k, (c, t) in sorted(per.items(), key=lambda x: -x[1][1]):
        lines.append(f"{k[:78]:78s} {c:6d} {t / c:9.1f} {t / a.steps:9.1f} {family(k)}")
    lines.append("")
    lines.append("per family, a launch per bin on one stream (ms per iteration): " +
                 ", ".join(f"{f} {v:.3f}" for f, v in sorted(fam.items(), key=lambda x: -x[1])))
    out = {"workload": a.workload, "K": a.K, "steps": a.steps, "ms_per_iter": dict(fam)}
    if a.fetch and a.write:
        ps = a.pmc_steps or a.steps
        fetch, cf = counter_summary(a.fetch, "FETCH_SIZE", ps)
        write, cw = counter_summary(a.write, "WRITE_SIZE", ps)
        ff = COPY_BYTES / (sum(cf) / len(cf)) if cf else 1.0
        fw = COPY_BYTES / (sum(cw) / len(cw)) if cw else 1.0
        lines.append("")
        lines.append(f"copy calibration (256 MiB k_calibration_copy): FETCH_SIZE factor {ff:.3f}, WRITE_SIZE factor {fw:.3f}"
                     f" ({len(cf)} / {len(cw)} copies)")
        lines.append(f"{'family':10s} {'fetch MB/iter':>14s} {'write MB/iter':>14s} {'HBM GB/s':>10s}")
        traffic = {}
        for f in sorted(set(fetch) | set(write)):
            fb, wb = fetch.get(f, 0.0) * ff, write.get(f, 0.0) * fw
            ms = fam.get(f, 0.0)
            gbs = (fb + wb) / (ms / 1e3) / 1e9 if ms else 0.0
            traffic[f] = {"fetch_bytes": fb, "write_bytes": wb, "ms": ms}
            lines.append(f"{f:10s} {fb / 1e6:14.1f} {wb / 1e6:14.1f} {gbs:10.1f}")
        out["traffic_per_iter"] = traffic
        out["copy_factor"] = {"fetch": ff, "write": fw}
    out["commands"] = [c.strip() for c in a.command.split(";") if c.strip()]
    with open(a.out + "_kernels.txt", "w") as f:
        f.write("\n".join(lines) + "\n")
    with open(a.out + "_traffic.json", "w") as f:
        json.dump(out, f, indent=1)
    print("\n".join(lines))


if __name__ == "__main__":
    main()
