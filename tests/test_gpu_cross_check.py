"""The FP64 general matvec and the residual norms against the kernels of a context made
under DEX_MATVEC=generic, which share nothing with them: cubes (NN=11), planes (NN=13, 17,
19, 21), planes with the intermediate in Y (NN=23, 25).

Bounds: 1e-13 of max|y| and of the norms (another summation order of the same products).
Two programs round apart, so some entries differ in their last bits; a context that ran
the same kernels twice would agree in every bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dex():
    import doublyexcited_amd as d

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return d


def _run(dex, n, x, e):
    with dex.HeliumGrid(n, 0.45, 0.3) as g:
        y = torch.full_like(x, float("nan"))
        g.matvec_device(x, y, 1)
        return y, g.residuals_device(x, e), g.fast_path


@pytest.mark.parametrize("n", [1, 2, 5, 6, 8, 9, 10, 11, 12])
def test_general_matvec_and_residuals_against_other_kernels(dex, monkeypatch, n):
    print(f"case: cross-check N={n}", flush=True)
    monkeypatch.delenv("DEX_MATVEC", raising=False)
    x = torch.randn((2 * n + 1) ** 6, dtype=torch.complex128, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(n))
    e = np.array([-0.7 - 0.02j])
    y, r, fast = _run(dex, n, x, e)
    assert fast == (n <= 10)
    monkeypatch.setenv("DEX_MATVEC", "generic")
    yg, rg, fast = _run(dex, n, x, e)
    assert not fast
    assert (y - yg).abs().max().item() <= 1e-13 * yg.abs().max().item()
    assert abs(r[0] - rg[0]) <= 1e-13 * rg[0]
    assert not torch.equal(y, yg)


def test_shifted_solve_on_the_other_kernels(dex, monkeypatch):
    """An inner solve of general vectors, whose matvecs take the shift.  Bound: the
    minimiser of one well-conditioned small problem, 1e-10 of its largest entry."""
    print("case: cross-check shift", flush=True)
    out = []
    for env in (None, "generic"):
        monkeypatch.delenv("DEX_MATVEC", raising=False)
        if env:
            monkeypatch.setenv("DEX_MATVEC", env)
        with dex.HeliumGrid(6, 0.5, 0.3) as g:
            x = torch.randn(2 * g.d, dtype=torch.complex128, device="cuda",
                            generator=torch.Generator(device="cuda").manual_seed(3))
            y = torch.empty_like(x)
            g.precblock_device(x, y, 2, 9.0 - 6.0j, 3)
            out.append(y)
    assert (out[0] - out[1]).abs().max().item() <= 1e-10 * out[1].abs().max().item()
    assert not torch.equal(out[0], out[1])


@pytest.mark.parametrize("n", [6, 11])
def test_launches_are_booked_by_the_kernels_that_run(dex, monkeypatch, n):
    """The planes' passes under pass1 and pass2, with the intermediate in Y (NN=23) and for
    residual norms too: 32 bytes an entry, then 96, or 80 where the last pass writes sums; a
    cross-check context's launches, 320 bytes an entry, under generic."""
    print(f"case: booked launches N={n}", flush=True)
    monkeypatch.delenv("DEX_MATVEC", raising=False)
    x = torch.randn((2 * n + 1) ** 6, dtype=torch.complex128, device="cuda")
    for env in (None, "generic"):
        if env:
            monkeypatch.setenv("DEX_MATVEC", env)
        with dex.HeliumGrid(n, 0.45, 0.3) as g:
            for call, rest in ((lambda: g.matvec_device(x, torch.empty_like(x), 1), 96),
                               (lambda: g.residuals_device(x, np.array([-0.7 + 0j])), 80)):
                g.reset_kernel_stats()
                call()
                t = {k: (v[0], v[1] / g.d) for k, v in g.kernel_totals().items() if v[0] and k != "coldots"}
                assert t == ({"generic": (1, 320)} if env else {"pass1": (1, 32), "pass2": (1, rest)})
