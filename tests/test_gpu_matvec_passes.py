"""The matvec's passes at the grids where they can go wrong: fewer points than a
transpose tile (NN=3), ragged tiles and tile blocks, one workgroup a CU (NN=21),
a batch of columns that ends inside a launch, output over the input.

Bounds: FP64 within 1e-13 of max|y| of the dense product (another summation order
of the same products), FP32 arithmetic within 2e-6."""
import math

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dex():
    import doublyexcited_amd as d

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return d


def _dense(g, x):
    """H x in FP64 from the grid's own tables: s2 (X K + K X) + c1 V o X on X[q, p]."""
    nn, m = g.nn, g.m
    t1 = torch.from_numpy(g.kematrix().copy()).cuda()
    one = torch.eye(nn, dtype=torch.float64, device="cuda")
    k3 = (torch.kron(one, torch.kron(one, t1)) + torch.kron(one, torch.kron(t1, one))
          + torch.kron(t1, torch.kron(one, one)))
    tab = torch.from_numpy(g.tinv().copy()).cuda()
    lab = torch.arange(m, device="cuda")
    ax = (lab % nn, lab // nn % nn, lab // nn ** 2)
    vn = -g.charge / g.delta ** 3 * tab[tuple(a - g.n + nn for a in ax)]
    v = vn[:, None] + vn[None, :] + tab[tuple(a[:, None] - a[None, :] + nn for a in ax)] / g.delta ** 3
    z = x.view(m, m).to(torch.complex128)
    zr, zi = z.real.contiguous(), z.imag.contiguous()
    k = torch.complex(zr @ k3 + k3 @ zr, zi @ k3 + k3 @ zi)
    s2 = complex(math.cos(2 * g.theta), -math.sin(2 * g.theta))
    c1 = complex(math.cos(g.theta), -math.sin(g.theta))
    return (s2 * k + c1 * v * z).reshape(-1)


def _block(g, cols, sym, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(cols, g.m, g.m, dtype=dtype, device="cuda", generator=gen)
    if sym:
        x = 0.5 * (x + sym * x.transpose(1, 2))
    return x.contiguous().view(-1)


@pytest.mark.parametrize("n,prec,single,sym,cols", [
    (1, "fp64", False, 1, 3), (1, "fp64", False, 0, 2), (2, "fp64", False, -1, 17), (2, "fp32", True, 1, 17),
    (3, "fp64", False, 0, 3), (4, "fp64", False, 1, 2), (4, "fp32", True, 0, 2), (4, "fp32", True, 0, 16),
    (4, "fp64", False, 0, 15), (5, "fp32", False, 0, 5), (6, "fp64", False, -1, 3),
    (6, "fp32", True, -1, 5), (6, "fp32", False, 1, 2), (6, "fp32", False, 0, 1), (7, "fp64", False, 0, 1),
    (8, "fp64", False, 1, 2), (9, "fp32", True, 1, 2), (10, "fp64", False, -1, 1), (11, "fp32", True, 1, 1),
    (11, "fp32", True, 0, 1), (11, "fp64", False, 0, 1), (12, "fp32", True, -1, 1), (12, "fp64", False, 0, 1)])
def test_passes_against_the_dense_product(dex, n, prec, single, sym, cols):
    print(f"case: passes N={n} {prec} complex64={single} sym={sym} cols={cols}", flush=True)
    with dex.HeliumGrid(n, 0.45, 0.3, precision=prec) as g:
        x = _block(g, cols, sym, torch.complex64 if single else torch.complex128, 10 * n + sym)
        y = torch.full_like(x, float("nan"))
        g.matvec_device(x, y, cols, single=single, symmetry=sym)
        tol = 1e-13 if prec == "fp64" else 2e-6
        for j in {0, cols - 1}:
            ref = _dense(g, x[j * g.d:(j + 1) * g.d])
            err = (y[j * g.d:(j + 1) * g.d].to(torch.complex128) - ref).abs().max().item()
            assert err <= tol * ref.abs().max().item(), (j, err)
        if sym:
            ym = y.view(cols, g.m, g.m)
            assert torch.equal(ym, sym * ym.transpose(1, 2))


@pytest.mark.parametrize("n,prec,single,sym,cols", [
    (2, "fp64", False, 1, 3), (5, "fp64", False, 0, 2), (5, "fp32", True, -1, 2), (5, "fp32", False, 1, 2),
    (8, "fp64", False, 0, 1)])
def test_output_over_the_input(dex, n, prec, single, sym, cols):
    """Y in X's own storage: bitwise the result in separate storage."""
    print(f"case: in place N={n} {prec} complex64={single} sym={sym} cols={cols}", flush=True)
    with dex.HeliumGrid(n, 0.45, 0.3, precision=prec) as g:
        x = _block(g, cols, sym, torch.complex64 if single else torch.complex128, n)
        y = torch.empty_like(x)
        g.matvec_device(x, y, cols, single=single, symmetry=sym)
        g.matvec_device(x, x, cols, single=single, symmetry=sym)
        assert torch.equal(x, y)


@pytest.mark.parametrize("n,prec,cols", [(3, "fp64", 3), (6, "fp64", 3), (6, "fp32", 130), (8, "fp64", 2),
                                         (11, "fp64", 1)])
def test_residuals_against_the_dense_product(dex, n, prec, cols):
    """||H x - e x|| / ||x|| within 1e-13 of the dense product's (sums of D squares
    of values that differ from the dense ones by 1e-15 of their largest)."""
    import numpy as np

    print(f"case: residuals N={n} {prec} cols={cols}", flush=True)
    with dex.HeliumGrid(n, 0.45, 0.3, precision=prec) as g:
        x = _block(g, min(cols, 3), 0, torch.complex128, n)
        x = x.repeat((cols + 2) // 3)[:cols * g.d].contiguous() if cols > 3 else x
        e = -0.7 + 0.01 * np.arange(cols) - 0.02j * np.arange(cols)
        got = g.residuals_device(x, e)
        for j in {0, cols // 2, cols - 1}:
            v = x[j * g.d:(j + 1) * g.d]
            ref = (torch.linalg.vector_norm(_dense(g, v) - complex(e[j]) * v) / torch.linalg.vector_norm(v)).item()
            assert abs(got[j] - ref) <= 1e-13 * ref, j


@pytest.mark.parametrize("n,sym", [(2, 0), (2, 1), (5, 1)])
def test_outputs_one_column_along_the_inputs(dex, n, sym):
    """Y one column along X: each column takes the product of the one before."""
    print(f"case: chained columns N={n} sym={sym}", flush=True)
    with dex.HeliumGrid(n, 0.45, 0.3) as g:
        buf = torch.zeros(4 * g.d, dtype=torch.complex128, device="cuda")
        buf[:g.d] = _block(g, 1, sym, torch.complex128, n)
        ref = [buf[:g.d].clone()]
        for _ in range(3):
            y = torch.empty_like(ref[-1])
            g.matvec_device(ref[-1], y, 1, symmetry=sym)
            ref.append(y)
        g.matvec_device(buf[:3 * g.d], buf[g.d:], 3, symmetry=sym)
        assert torch.equal(buf, torch.cat(ref))
