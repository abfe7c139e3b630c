"""Combinations at every output width of their kernels (1..4, ..8, ..12, ..16 in
registers, ..32 through LDS, ..48), through order-2 inner solves of as many columns.

The solve is the least-squares fit of the block by (H - sigma) [B, H B], done here by
a QR in FP64.  Bound: random columns make a well-conditioned fit (below 1e3), 1e-9 of
the largest entry."""
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


@pytest.mark.parametrize("n,cols,sym", [
    (1, 2, 0), (2, 1, 0), (2, 3, 1), (2, 5, 0), (2, 8, -1), (2, 11, 0), (2, 15, 1), (2, 17, 0), (2, 25, 1),
    (2, 33, 0), (2, 48, 0)])
def test_order_two_block_solve_is_the_least_squares_fit(dex, n, cols, sym):
    print(f"case: widths n={n} cols={cols} sym={sym}", flush=True)
    sigma = -0.7 - 0.002j
    with dex.HeliumGrid(n, 0.5, 0.3) as g:
        gen = torch.Generator(device="cuda").manual_seed(cols)
        b = torch.randn(cols, g.m, g.m, dtype=torch.complex128, device="cuda", generator=gen)
        b = (0.5 * (b + sym * b.transpose(1, 2)) if sym else b).contiguous().view(-1)
        x, hb, hhb = torch.empty_like(b), torch.empty_like(b), torch.empty_like(b)
        g.precblock_device(b, x, cols, sigma, 2, symmetry=sym)
        g.matvec_device(b, hb, cols, symmetry=sym)
        g.matvec_device(hb, hhb, cols, symmetry=sym)
        g.sync()
        got, b, hb, hhb = (v.view(cols, g.d).cpu().numpy().T for v in (x, b, hb, hhb))
    basis = np.hstack([b, hb])
    scale = np.linalg.norm(basis, axis=0)
    q, r = np.linalg.qr(np.hstack([hb - sigma * b, hhb - sigma * hb]) / scale)
    ref = (basis / scale) @ np.linalg.solve(r, q.conj().T @ b)
    assert np.max(np.abs(got - ref)) <= 1e-9 * np.max(np.abs(ref))
