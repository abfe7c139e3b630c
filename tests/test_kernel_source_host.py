"""Rules of the kernel source that no run on a device shows reliably."""
import re
from pathlib import Path

SOURCE = Path(__file__).resolve().parents[1] / "doublyexcited_amd" / "csrc" / "dex_kernels.hip"


def _kernels():
    """(name, parameters, body) of every __global__ function."""
    text = re.sub(r"//[^\n]*", "", SOURCE.read_text())

    def closing(at, pair):  # the index behind the bracket that closes the one at `at`
        depth = 0
        for i in range(at, len(text)):
            depth += (text[i] == pair[0]) - (text[i] == pair[1])
            if depth == 0:
                return i + 1
        raise AssertionError("unbalanced brackets")

    for g in re.finditer(r"__global__", text):
        head = re.compile(r"\b(k_\w+)\s*\(").search(text, g.end())
        end = closing(head.end() - 1, "()")
        body = text.index("{", end)
        yield head.group(1), text[head.end():end - 1], text[body:closing(body, "{}")]


def test_a_thread_leaves_a_kernel_only_behind_its_barriers():
    """A return before a __syncthreads() takes the whole workgroup: its condition is of
    blockIdx alone (a tile pair beyond the matrix, the lower triangle of tiles)."""
    uniform = ("!sym_tile(m, nblk, ta, tb)", "bi > bj")
    seen = 0
    for name, _, body in _kernels():
        before = body[:body.rfind("__syncthreads()")] if "__syncthreads()" in body else ""
        for r in re.finditer(r"if \((.*)\)\s*return;", before):
            seen += 1
            assert r.group(1) in uniform, (name, r.group(0))
    assert seen >= 3  # k_symfold, k_combine_sym, k_singlet


def test_arrays_that_may_be_one_are_not_declared_apart():
    """Kernels whose callers pass one array as input and output declare neither
    __restrict__: the general second passes (Y over X or Z) and the projection (Y over X)."""
    shared = {"k_pass2": ("x", "z", "y"), "k_plane2": ("x", "z", "y"), "k_singlet": ("x", "y")}
    got = {name: params for name, params, _ in _kernels() if name in shared}
    assert set(got) == set(shared)
    for name, arrays in shared.items():
        for a in arrays:
            assert re.search(rf"\*\s*{a}\b", got[name]), (name, a)
            assert not re.search(rf"__restrict__\s+{a}\b", got[name]), (name, a)


def test_every_kernel_has_its_class_in_the_profile_tools():
    """A kernel without a class drops out of the class table and the traffic ratios; a class
    entry without a kernel is stale."""
    from doublyexcited_amd import _lib, profsummary

    names = {name for name, _, _ in _kernels()}
    assert set(profsummary.CLASSES) | set(profsummary.UNCLASSED) == names
    assert not set(profsummary.CLASSES) & set(profsummary.UNCLASSED)
    assert {c for c, _ in profsummary.CLASSES.values()} == set(_lib.KERNEL_CLASSES)
    for name, (cls, share) in profsummary.CLASSES.items():
        full = f"void dex::(anonymous namespace)::{name}<21, double, HIP_vector_type<double, 2u>, false>(dex::Arg, int)"
        assert profsummary.kernel_class(full) == (cls, share)
