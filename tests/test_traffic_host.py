"""The HBM-traffic analysis of two rocprofv3 counter passes (host logic only):
calibration scaling and per-class traffic / algorithmic ratios."""
import json

import pytest

from doublyexcited_amd.profsummary import class_table
from doublyexcited_amd.traffic import analyse

HDR = "Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value\n"


def _write(d, counter, rows):
    d.mkdir(parents=True, exist_ok=True)
    (d / "run_counter_collection.csv").write_text(
        HDR + "".join(f'{i},"{n}",{counter},{v}\n' for i, n, v in rows))


def test_ratios_from_calibrated_counters(tmp_path):
    gib_kib = (1 << 30) / 1024.0
    ns = "void dex::(anonymous namespace)::"
    # torch's fill, then the calibration multiply: FETCH reports half of the bytes read, WRITE all
    # of them (the fill writes as much and reads nothing)
    fill = "void at::native::vectorized_elementwise_kernel<4, at::native::FillFunctor<c10::complex<double> > >(int)"
    mul = "void at::native::vectorized_elementwise_kernel<4, at::native::AUnaryFunctor<c10::complex<double> > >(int)"
    fetch = [(1, fill, 20.0), (2, mul, gib_kib / 2)]
    write = [(1, fill, gib_kib), (2, mul, gib_kib)]
    # a library kernel outside the classes with a larger count must not be taken for the calibration
    fetch.append((3, "dex::(anonymous namespace)::k_singlet(HIP_vector_type<double, 2u>*, long, double)", 4 * gib_kib))
    write.append((3, "dex::(anonymous namespace)::k_singlet(HIP_vector_type<double, 2u>*, long, double)", 2 * gib_kib))
    # two combine launches, each reading 2 GB and writing 1 GB (FETCH at half scale)
    for i in (4, 5):
        fetch.append((i, ns + "k_combine_w<12, 2, 8>(dex::ColDesc const*, int, int)", 2e9 / 1024 / 2))
        write.append((i, ns + "k_combine_w<12, 2, 8>(dex::ColDesc const*, int, int)", 1e9 / 1024))
    # one Gram launch reading 1 GB, and its partial-sum reduction reading 1 MB
    fetch += [(6, ns + "k_gram_mfma<2, 1, 32>(dex::ColDesc const*, int)", 1e9 / 1024 / 2),
              (7, "dex::(anonymous namespace)::k_reduce_partials(HIP_vector_type<double, 2u> const*, int)",
               1e6 / 1024 / 2)]
    write += [(6, ns + "k_gram_mfma<2, 1, 32>(dex::ColDesc const*, int)", 0.0),
              (7, "dex::(anonymous namespace)::k_reduce_partials(HIP_vector_type<double, 2u> const*, int)", 0.0)]
    # a column-dot launch and a residual step (both coldots launches), each reading 1 GB and writing
    # 0.5 GB with its reduction
    for i, k in ((8, "k_coldots(dex::ColDesc const*, int, long, double*)"),
                 (9, "k_resid(dex::ColDesc const*, int, double const*)")):
        fetch.append((i, "dex::(anonymous namespace)::" + k, 1e9 / 1024 / 2))
        write.append((i, "dex::(anonymous namespace)::" + k, 0.5e9 / 1024))
    _write(tmp_path / "f", "FETCH_SIZE", fetch)
    _write(tmp_path / "w", "WRITE_SIZE", write)
    stats = tmp_path / "stats.json"
    # algorithmic: combine 3 GB per launch, Gram 0.9 GB per launch, coldots 1.5 GB per launch
    stats.write_text(json.dumps({"totals": {"combine": [2, 6e9, 0], "gram": [1, 0.9e9, 0],
                                            "coldots": [2, 3e9, 0]}}))
    cf, cw, fs, ws, table, ratios = analyse(tmp_path / "f", tmp_path / "w", stats)
    assert abs(fs - 2.0) < 1e-12 and abs(ws - 1.0) < 1e-12
    assert abs(ratios["combine"] - 1.0) < 1e-9
    assert abs(ratios["gram"] - (1e9 + 1e6) / 0.9e9) < 1e-9
    assert abs(ratios["coldots"] - 1.0) < 1e-9
    assert {row[0]: row[1] for row in table} == {"combine": 2, "gram": 1, "coldots": 2}


NS = "void dex::(anonymous namespace)::"
MUL = "void at::native::vectorized_elementwise_kernel<4, at::native::AUnaryFunctor<c10::complex<double> > >(int)"


def _passes(tmp_path, kernels, totals):
    """Counter passes of one dispatch per (kernel, GB read, GB written)."""
    gib_kib = (1 << 30) / 1024.0
    rows = [(i + 2, NS + k + "(int)", r, w) for i, (k, r, w) in enumerate(kernels)]
    _write(tmp_path / "f", "FETCH_SIZE", [(1, MUL, gib_kib / 2)] + [(i, k, r * 1e9 / 2048) for i, k, r, _ in rows])
    _write(tmp_path / "w", "WRITE_SIZE", [(1, MUL, gib_kib)] + [(i, k, w * 1e9 / 1024) for i, k, _, w in rows])
    stats = tmp_path / "stats.json"
    stats.write_text(json.dumps({"totals": totals}))
    return analyse(tmp_path / "f", tmp_path / "w", stats)


def test_matvec_passes_fall_into_their_classes(tmp_path):
    """The transpose-add, the planes (two dispatches of the remaining passes a launch, with a
    reduction for norms) and a cross-check context's seven launches."""
    kernels = [("k_pass1<21, double, HIP_vector_type<double, 2u>, false>", 1.0, 1.0),
               ("k_symfold<HIP_vector_type<double, 2u> >", 1.0, 1.0),
               ("k_plane1<25, double>", 1.0, 1.0), ("k_plane2<25, double, false>", 2.0, 1.0),
               ("k_plane2<25, double, true>", 2.0, 0.0), ("k_reduce_wide", 0.5, 0.0)]
    kernels += [("k_axis<5>", 1.0, 1.0)] * 6 + [("k_potential", 2.0, 1.0)]
    *_, table, ratios = _passes(tmp_path, kernels, {
        "pass1": [2, 4e9, 0], "symadd": [1, 2e9, 0], "pass2": [1, 5.5e9, 0], "generic": [1, 15e9, 0],
        "combine": [0, 0.0, 0]})
    assert {row[0]: row[1] for row in table} == {"pass1": 2, "symadd": 1, "pass2": 1, "generic": 1}
    assert all(abs(r - 1.0) < 1e-9 for r in ratios.values()) and len(ratios) == 4


def test_a_class_without_its_kernels_is_an_error(tmp_path):
    with pytest.raises(SystemExit, match="symadd.*k_renamed"):
        _passes(tmp_path, [("k_renamed", 1.0, 1.0)], {"symadd": [3, 6e9, 0]})


def test_class_table_counts_launches_and_names_what_has_no_class():
    rows = [{"Name": NS + k + "(int)", "Calls": str(n), "TotalDurationNs": str(t)} for k, n, t in (
        ("k_symfold<float>", 4, 4e6), ("k_plane1<13, double>", 3, 3e6), ("k_plane2<13, double, false>", 6, 12e6),
        ("k_singlet", 2, 1e6))]
    rows.append({"Name": MUL, "Calls": "9", "TotalDurationNs": "9e6"})
    assert class_table(rows)[2:] == ["| pass2 | 3 | 12.0 | 4000.0 |", "| symadd | 4 | 4.0 | 1000.0 |",
                                     "| pass1 | 3 | 3.0 | 1000.0 |", "| (no class) | 2 | 1.0 | 500.0 |"]
