"""HBM traffic per kernel launch from two rocprofv3 counter passes.

Usage::

    python -m doublyexcited_amd.traffic FETCH_DIR WRITE_DIR STATS_JSON [OUT_JSON]

``FETCH_DIR`` and ``WRITE_DIR`` hold the ``*counter_collection.csv`` of a
``rocprofv3 --pmc FETCH_SIZE`` and a ``rocprofv3 --pmc WRITE_SIZE`` run of the
same program (``bench.py --traffic-run STATS_JSON ...``), which first runs a
calibration kernel (an elementwise multiply that reads and writes 1 GiB) and
then the profiled solve, whose per-class algorithmic bytes and launch counts it
writes to ``STATS_JSON``.  The calibration dispatch scales each counter to
bytes (FETCH_SIZE reports half of the bytes read on this part); per kernel
class the scaled traffic per launch is divided by the algorithmic bytes per
launch.  A class with launches but no kernel of its own in the passes is an
error.  Prints a Markdown table and writes ``{"traffic_over_algorithmic":
{class: ratio}}`` to ``OUT_JSON`` when given.
"""
from __future__ import annotations

import csv
import json
import sys
from pathlib import Path

from .profsummary import base, kernel_class

CAL_BYTES = 1 << 30  # the calibration kernel reads and writes 1 GiB


def _rows(d: Path, counter: str):
    files = sorted(Path(d).rglob("*counter_collection.csv"))
    if not files:
        raise SystemExit(f"no counter_collection.csv under {d}")
    out = []
    for f in files:
        with open(f, newline="") as fh:
            for r in csv.DictReader(fh):
                if r.get("Counter_Name") == counter:
                    out.append((r.get("Kernel_Name", ""), int(r.get("Dispatch_Id", 0)), float(r["Counter_Value"])))
    return out


def _per_dispatch(rows):
    acc = {}
    for name, disp, val in rows:
        k = (name, disp)
        acc[k] = acc.get(k, 0.0) + val
    return acc


def analyse(fetch_dir, write_dir, stats_json):
    fetch = _per_dispatch(_rows(fetch_dir, "FETCH_SIZE"))
    write = _per_dispatch(_rows(write_dir, "WRITE_SIZE"))
    # calibration: the elementwise multiply, the largest counter value among torch's kernels
    # (the fill before it writes as much and reads nothing)
    def cal(acc):
        cands = [v for (n, d), v in acc.items() if "at::native" in n and v > 0]
        return max(cands) if cands else None
    cf, cw = cal(fetch), cal(write)
    f_scale = CAL_BYTES / (cf * 1024.0)
    w_scale = CAL_BYTES / (cw * 1024.0)
    stats = json.loads(Path(stats_json).read_text())
    totals = stats.get("totals", stats)
    table = []
    ratios = {}
    for c, (launches, alg_bytes, *_) in totals.items():
        if launches <= 0:
            continue
        # the class's kernels, the helpers that finish a launch (partial-sum reductions) among them
        fv = [(n, v) for (n, _), v in fetch.items() if kernel_class(n)[0] == c]
        wv = [(n, v) for (n, _), v in write.items() if kernel_class(n)[0] == c]
        nf, nw = (sum(kernel_class(n)[1] for n, _ in x) for x in (fv, wv))
        if nf <= 0 or nw <= 0:
            raise SystemExit(f"class {c}: {launches} launches in {stats_json}, but none of its kernels in the "
                             f"counter passes (kernels seen: {sorted({base(n) for n, _ in fetch})})")
        f, w = sum(v for _, v in fv) / nf, sum(v for _, v in wv) / nw
        traffic = (f * f_scale + w * w_scale) * 1024.0
        alg = alg_bytes / launches
        ratios[c] = traffic / alg
        table.append((c, nf, f, w, traffic / 1e9, alg / 1e9, traffic / alg))
    return cf, cw, f_scale, w_scale, table, ratios


def main(argv=None) -> int:
    argv = sys.argv[1:] if argv is None else argv
    if len(argv) < 3:
        print(__doc__)
        return 2
    cf, cw, fs, ws, table, ratios = analyse(argv[0], argv[1], argv[2])
    print(f"Calibration (1 GiB read + 1 GiB written): FETCH_SIZE {cf:.1f} KiB, WRITE_SIZE {cw:.1f} KiB; "
          f"scale FETCH x {fs:.4f}, WRITE x {ws:.4f}\n")
    print("| class | launches | FETCH_SIZE KiB/launch | WRITE_SIZE KiB/launch | scaled traffic GB/launch "
          "| algorithmic GB/launch | traffic / algorithmic |")
    print("|---|---:|---:|---:|---:|---:|---:|")
    for c, n, f, w, t, a, r in table:
        print(f"| {c} | {n:g} | {f:.1f} | {w:.1f} | {t:.4f} | {a:.4f} | {r:.3f} |")
    if len(argv) > 3:
        Path(argv[3]).write_text(json.dumps({"source": argv[2], "traffic_over_algorithmic": ratios}, indent=1))
    return 0


if __name__ == "__main__":
    sys.exit(main())
