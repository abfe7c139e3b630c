"""The inner solve's shifted matvec on each of its routes: cubes (NN=9, general and
symmetric), planes (NN=13) and symmetric cubes of one workgroup a CU (NN=19).

An order-2 solve of one column is the least-squares fit of b by the two vectors
(H - sigma) b and (H - sigma) H b, formed here with the plain matvec; with |sigma| of
the order of H's spectrum a wrong shift shows at once.  Bound: the fit's 2 x 2 normal
equations in FP64 at condition numbers below 1e4, 1e-10 of the largest entry."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dex():
    import doublyexcited_amd as d

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return d


@pytest.mark.parametrize("n,sym", [(4, 0), (4, 1), (6, 0), (6, -1), (9, 1)])
@pytest.mark.parametrize("sigma", [-0.7 - 0.002j, 9.0 - 6.0j])
def test_order_two_solve_is_the_two_vector_fit(dex, n, sym, sigma):
    print(f"case: shift n={n} sym={sym} sigma={sigma}", flush=True)
    with dex.HeliumGrid(n, 0.5, 0.3) as g:
        gen = torch.Generator(device="cuda").manual_seed(n)
        b = torch.randn(g.m, g.m, dtype=torch.complex128, device="cuda", generator=gen)
        b = (0.5 * (b + sym * b.T) if sym else b).contiguous().view(-1)
        x, hb, hhb = torch.empty_like(b), torch.empty_like(b), torch.empty_like(b)
        g.precblock_device(b, x, 1, sigma, 2, symmetry=sym)
        g.matvec_device(b, hb, symmetry=sym)
        g.matvec_device(hb, hhb, symmetry=sym)
        g.sync()
        basis = [b, hb]
        image = [hb - sigma * b, hhb - sigma * hb]
        k = torch.tensor([[torch.vdot(u, v).item() for v in image] for u in image], dtype=torch.complex128)
        r = torch.tensor([torch.vdot(u, b).item() for u in image], dtype=torch.complex128)
        y = torch.linalg.solve(k, r)
        ref = y[0].item() * basis[0] + y[1].item() * basis[1]
        assert (x - ref).abs().max().item() <= 1e-10 * ref.abs().max().item()
