"""Markdown summary of a rocprofv3 ``--kernel-trace --stats`` run.

Usage::

    python -m doublyexcited_amd.profsummary STATS_CSV [TITLE] [COMMAND]

``STATS_CSV`` is the ``*kernel_stats.csv`` rocprofv3 writes with ``-f csv``.
Prints the total kernel time and, per kernel, calls, total and average
duration and share, largest first; kernel names are shortened to the
library's template names.
"""
from __future__ import annotations

import csv
import re
import sys


def short(name: str) -> str:
    n = re.sub(r"dex::\(anonymous namespace\)::", "", name)
    n = re.sub(r"HIP_vector_type<(\w+), \d+u>", r"\1x", n)
    n = re.sub(r"\(.*\)$", "", n).strip()
    return n


# kernel -> (the library's kernel class, launches of the class that one dispatch of the
# kernel is).  A Gram is its partial kernel and the partial-sum reduction, a residual
# step its kernel and a reduction, the planes' remaining passes two dispatches (the last
# followed by a reduction where it forms residual norms), a general matvec of a
# cross-check context six axes and the potential.
CLASSES = {
    "k_pass1": ("pass1", 1.0), "k_plane1": ("pass1", 1.0), "k_direct": ("pass1", 1.0),
    "k_pass2": ("pass2", 1.0), "k_plane2": ("pass2", 0.5), "k_reduce_wide": ("pass2", 0.0),
    "k_symfold": ("symadd", 1.0),
    "k_gram_mfma": ("gram", 1.0), "k_gram_pk": ("gram", 1.0), "k_reduce_partials": ("gram", 0.0),
    "k_combine": ("combine", 1.0), "k_combine_w": ("combine", 1.0), "k_combine_sym": ("combine", 1.0),
    "k_coldots": ("coldots", 1.0), "k_resid": ("coldots", 1.0), "k_reduce_real": ("coldots", 0.0),
    "k_axis": ("generic", 0.0), "k_potential": ("generic", 1.0),
}
# kernels outside the classes: start vectors, projections, conversions, the one-electron
# Lanczos and the orbital subspace
UNCLASSED = ("k_fill_gaussian", "k_singlet", "k_to_single", "k_to_double", "k_h1", "k_small_dots",
             "k_small_lincomb", "k_lowrank", "k_ywx")


def base(name: str) -> str:
    """A kernel's own name: no return type, namespaces, template or parameter list."""
    n = name.replace("(anonymous namespace)::", "")
    return n.split("<")[0].split("(")[0].replace("void ", "").strip().split("::")[-1]


def kernel_class(name: str):
    """(class, launches of it that a dispatch is); (None, 0.0) outside the classes."""
    return CLASSES.get(base(name), (None, 0.0))


def class_table(rows) -> list[str]:
    tot = {}
    for r in rows:
        cls, share = kernel_class(r["Name"])
        if cls is None:
            if not base(r["Name"]).startswith("k_"):
                continue  # another library's
            cls, share = "(no class)", 1.0
        t, n = tot.get(cls, (0.0, 0.0))
        tot[cls] = (t + float(r["TotalDurationNs"]), n + share * int(r["Calls"]))
    out = ["| class | launches | total ms | avg us per launch |", "|---|---:|---:|---:|"]
    for cls, (t, n) in sorted(tot.items(), key=lambda kv: -kv[1][0]):
        out.append(f"| {cls} | {n:g} | {t / 1e6:.1f} | {t / n / 1e3 if n else 0.0:.1f} |")
    return out


def summarize(path: str, title: str = "", command: str = "") -> str:
    rows = list(csv.DictReader(open(path, newline="")))
    tot = sum(float(r["TotalDurationNs"]) for r in rows)
    calls = sum(int(r["Calls"]) for r in rows)
    out = []
    if title:
        out.append(f"# {title}\n")
    if command:
        out.append("```\n" + command + "\n```\n")
    out.append(f"Total kernel time {tot / 1e9:.3f} s over {calls} dispatches.\n")
    out.append("| kernel | calls | total ms | avg us | % |")
    out.append("|---|---:|---:|---:|---:|")
    for r in sorted(rows, key=lambda r: -float(r["TotalDurationNs"])):
        t = float(r["TotalDurationNs"])
        if t < 0.001 * tot:
            continue
        out.append(f"| `{short(r['Name'])}` | {r['Calls']} | {t / 1e6:.1f} | {float(r['AverageNs']) / 1e3:.1f} | "
                   f"{100.0 * t / tot:.2f} |")
    out.append("")
    out.append("Per kernel class (the library's launch-statistics classes; a Gram launch includes its "
               "partial-sum reduction, a plane matvec's remaining passes are one launch):\n")
    out.extend(class_table(rows))
    return "\n".join(out) + "\n"


def main(argv=None) -> int:
    argv = sys.argv[1:] if argv is None else argv
    if not argv:
        print(__doc__)
        return 2
    print(summarize(argv[0], argv[1] if len(argv) > 1 else "", argv[2] if len(argv) > 2 else ""))
    return 0


if __name__ == "__main__":
    sys.exit(main())
