"""Summaries of rocprofv3 CSV output for the profiles of this package.

Usage:
  python -m cm1_amd.profsum trace <run_kernel_stats.csv>   # per-kernel time table
  python -m cm1_amd.profsum pmc <fetch counter csv> <write counter csv>
      # per-dispatch HBM bytes, calibrated on the plain copies that
      # ``bench.py --copy-calibration`` runs first (1 GiB each)

Kernel names are shortened to the device function each launcher runs
(``k_one<NT, F>`` and ``k_one_w<NT, W, F>``: ``F``'s host function and
lambda number)."""
import csv
import re
import sys
from collections import defaultdict


def short(name):
    """k_one<256, for3<cm1g_solve2::{lambda(int, int, int)#1}>(...)> -> for3<cm1g_solve2 λ1>."""
    m = re.match(r"void k_one(?:_w)?<\d+, (?:\d+, )?(.*)>\(", name)
    if not m:
        return name.split("(")[0]
    body = m.group(1).replace("(anonymous namespace)::", "")
    # for3<host::{lambda ...#n}>(...)::{lambda#1}  or  host(...)::{lambda(...)#n}
    f = re.match(r"(for[23])<([\w:]+?(?:<\d+>)?)(?:\(.*?\))?::\{lambda\(int, int(?:, int)?\)#(\d+)\}", body)
    if f:
        return f"{f.group(1)}<{f.group(2).split('::')[-1]} λ{f.group(3)}>"
    t = re.match(r"(\w+)<([^>]*)>\(", body)
    if t and t.group(1) == "slab_go":
        return "sound_slab"
    if t and t.group(1) in ("advs_launch", "advm_launch"):
        return {"advs_launch": "advs_col", "advm_launch": "advm_col"}[t.group(1)] + f"<{t.group(2)}>"
    h = re.match(r"([\w:]+)(?:\(.*?\))?::\{lambda\(int, int(?:, int)?\)#(\d+)\}", body)
    if h:
        host = h.group(1).split("::")[-1]
        names = {("sound_run", "1"): "sound_coef", ("sound_run", "2"): "sound_sub",
                 ("advs_run", "1"): "pdef_fix", ("cm1g_solve2", "2"): "massflux_div",
                 ("sounde_run", "2"): "sounde_col", ("sounde_run", "3"): "sounde_col"}
        if host == "kess_cols_run":
            return "kess_cols"
        return names.get((host, h.group(2)), f"{host} λ{h.group(2)}")
    return body.split("(")[0]


def trace(path):
    # the variants of a kernel that share a short name are one row
    per = defaultdict(lambda: [0, 0.0])
    for r in csv.DictReader(open(path)):
        e = per[short(r["Name"])]
        e[0] += int(r["Calls"])
        e[1] += float(r["TotalDurationNs"])
    tot = sum(ns for _, ns in per.values())
    print("| kernel | dispatches | total ms | avg us | share |")
    print("|---|---:|---:|---:|---:|")
    for name, (calls, ns) in sorted(per.items(), key=lambda e: -e[1][1]):
        print(f"| `{name}` | {calls} | {ns / 1e6:.2f} | {ns / calls / 1e3:.1f} | {100.0 * ns / tot:.1f}% |")
    print(f"\nWhole process kernel time {tot / 1e6:.1f} ms.")


def counters(path):
    """Values per kernel, the variants that share a short name together, and the model's own kernels."""
    per, model = defaultdict(list), set()
    for r in csv.DictReader(open(path)):
        n = r["Kernel_Name"]
        if "k_one" in n:
            n = short(n)
            model.add(n)
        per[n].append(float(r["Counter_Value"]))
    return per, model


def pmc(fpath, wpath):
    (f, model), (w, _) = counters(fpath), counters(wpath)
    gib = 1024.0 ** 3
    # calibration: the copies of 1 GiB the bench ran first
    cf = [v for n, vs in f.items() if "copyBuffer" in n for v in vs if v * 1024 > 0.25 * gib]
    cw = [v for n, vs in w.items() if "copyBuffer" in n for v in vs if v * 1024 > 0.5 * gib]
    rf = (gib / (min(cf) * 1024)) if cf else 1.0
    rw = (gib / (min(cw) * 1024)) if cw else 1.0
    print(f"Calibration: a plain device copy of 1 GiB reads FETCH_SIZE {min(cf) * 1024 / gib:.3f} GiB and "
          f"WRITE_SIZE {min(cw) * 1024 / gib:.3f} GiB, so bytes = FETCH_SIZE x {rf:.3f} + WRITE_SIZE x {rw:.3f} "
          f"(KiB counters x 1024).\n")
    rows = []
    for n in f:
        if n not in w or n not in model:
            continue
        rd = sum(f[n]) / len(f[n]) * 1024 * rf / 1e9
        wr = sum(w[n]) / len(w[n]) * 1024 * rw / 1e9
        rows.append((n, len(f[n]), rd, wr))
    print("| kernel | dispatches | read GB | write GB | traffic GB / dispatch |")
    print("|---|---:|---:|---:|---:|")
    for n, c, rd, wr in sorted(rows, key=lambda r: -(r[2] + r[3])):
        if rd + wr < 0.05:
            continue
        print(f"| `{n}` | {c} | {rd:.3f} | {wr:.3f} | {rd + wr:.3f} |")
    for n, c, rd, wr in rows:
        if n in ("sound_slab", "sound_sub"):
            print(f"\ntraffic {n} bytes_per_launch={(rd + wr) * 1e9:.1f}")


if __name__ == "__main__":
    if sys.argv[1] == "trace":
        trace(sys.argv[2])
    else:
        pmc(sys.argv[2], sys.argv[3])
