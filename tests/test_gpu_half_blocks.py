"""Block operations that read one half of exchange-symmetric vectors (NN >= 11),
against the same solve with every row read.

NN=11 has M = 1331 = 20 blocks of 64 and 51 rows (41 of 32 and 19), NN=13 M = 2197 =
34 blocks of 64 and 21 rows (68 of 32 and 21): ragged last blocks and odd columns.  The
widths take each of the combination's output counts (1..4, ..8, ..12, ..16) and one
above them, whose combinations read every row; order 8 of 9 columns passes the inputs
of one launch.  Bound: both are the minimiser of one well-conditioned small problem
from FP64 sums in another order, 1e-10 of the largest entry."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dex():
    import doublyexcited_amd as d

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return d


def _block(g, cols, sym, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(cols, g.m, g.m, dtype=torch.complex128, device="cuda", generator=gen)
    return (0.5 * (x + sym * x.transpose(1, 2))).contiguous().view(-1)


@pytest.mark.parametrize("n,cols,sym,order", [
    (5, 1, 1, 2), (5, 3, -1, 3), (5, 6, 1, 3), (5, 9, -1, 8), (5, 13, 1, 3), (5, 17, 1, 2), (6, 4, -1, 4),
    (6, 10, 1, 3)])
def test_inner_solve_by_halves(dex, n, cols, sym, order):
    print(f"case: halves n={n} cols={cols} sym={sym} order={order}", flush=True)
    with dex.HeliumGrid(n, 0.5, 0.3) as g:
        x = _block(g, cols, sym, 40 * n + cols)
        half, whole = torch.empty_like(x), torch.empty_like(x)
        g.precblock_device(x, half, cols, -0.7 - 0.002j, order, symmetry=sym)
        g.precblock_device(x, whole, cols, -0.7 - 0.002j, order, symmetry=0)
        assert (half - whole).abs().max().item() <= 1e-10 * whole.abs().max().item()
        h = half.view(cols, g.m, g.m)
        assert torch.equal(h, sym * h.transpose(1, 2))


def test_inner_solve_of_other_vectors_is_that_of_their_symmetric_part(dex):
    print("case: halves of other vectors", flush=True)
    with dex.HeliumGrid(5, 0.5, 0.3) as g:
        gen = torch.Generator(device="cuda").manual_seed(5)
        x = torch.randn(2, g.m, g.m, dtype=torch.complex128, device="cuda", generator=gen)
        xs = (0.5 * (x + x.transpose(1, 2))).contiguous().view(-1)
        x = x.view(-1)
        y, ys = torch.empty_like(x), torch.empty_like(x)
        g.precblock_device(x, y, 2, -0.7 - 0.002j, 3, symmetry=1)
        g.precblock_device(xs, ys, 2, -0.7 - 0.002j, 3, symmetry=1)
        assert (y - ys).abs().max().item() <= 1e-10 * ys.abs().max().item()


@pytest.mark.parametrize("sym,cols", [(1, 4), (-1, 3)])
def test_single_precision_basis_by_halves(dex, sym, cols):
    """complex64 columns (odd rows: pairs are 8-byte aligned): the Ritz values of two
    iterations with a complex64 inner basis, by halves and with every row read.  Both
    round at FP32's 6e-8, times |H| ~ 100 at most: 1e-5."""
    print(f"case: halves c64 sym={sym} cols={cols}", flush=True)
    with dex.HeliumGrid(5, 0.5, 0.3) as g:
        start = _block(g, cols, sym, 60 + cols)
        e = []
        for symmetry in (sym, 0):
            x = start.clone()
            e.append(g.gplmr_eig_device(x, -0.7 - 0.002j, cols, maxit=2, tol=1e-7, symmetry=symmetry, inner_iter=8,
                                        inner_fp32=True).e)
        assert abs(e[0] - e[1]).max() <= 1e-5


@pytest.mark.parametrize("n,cols,sym", [(2, 1, 1), (2, 17, -1), (5, 3, 1), (6, 2, -1)])
def test_order_one_of_other_vectors_is_that_of_their_symmetric_part(dex, n, cols, sym):
    """Order 1 is H X: for X of no symmetry H of its (anti)symmetric part, by the general
    passes here.  Bound: the same products in another summation order, 1e-13 of max|y|."""
    print(f"case: order 1 of other vectors n={n} cols={cols} sym={sym}", flush=True)
    with dex.HeliumGrid(n, 0.5, 0.3) as g:
        gen = torch.Generator(device="cuda").manual_seed(70 + n)
        x = torch.randn(cols, g.m, g.m, dtype=torch.complex128, device="cuda", generator=gen)
        xs = (0.5 * (x + sym * x.transpose(1, 2))).contiguous().view(-1)
        x = x.view(-1)
        kept, y, ref = x.clone(), torch.full_like(x, float("nan")), torch.empty_like(x)
        g.precblock_device(x, y, cols, -0.7 - 0.002j, 1, symmetry=sym)
        assert torch.equal(x, kept)
        # general passes one column at a time, outputs over the inputs: two launches at every grid
        ref.copy_(xs)
        for j in range(cols):
            v = ref[j * g.d:(j + 1) * g.d]
            g.matvec_device(v, v, 1)
        assert (y - ref).abs().max().item() <= 1e-13 * ref.abs().max().item()
