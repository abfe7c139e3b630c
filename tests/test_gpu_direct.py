"""General vectors of the smallest grids (NN = 3 and 5) in one launch, and in two where
the outputs lie over the inputs, against the dense-table oracle.

Bounds: FP64 within 1e-13 of max|y| (another summation order of the same products),
FP32 arithmetic within 2e-6."""
import numpy as np
import pytest

from oracle.hamiltonian import Hamiltonian

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dex():
    import doublyexcited_amd as d

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return d


@pytest.mark.parametrize("n", [1, 2])
@pytest.mark.parametrize("prec,single", [("fp64", False), ("fp32", True), ("fp32", False)])
@pytest.mark.parametrize("cols", [1, 3, 17])
def test_one_launch_and_two_against_the_oracle(dex, n, prec, single, cols):
    print(f"case: direct n={n} {prec} complex64={single} cols={cols}", flush=True)
    h = Hamiltonian(n, 0.45, 0.3)
    with dex.HeliumGrid(n, 0.45, 0.3, precision=prec) as g:
        gen = torch.Generator(device="cuda").manual_seed(n + cols)
        x = torch.randn(cols * g.d, dtype=torch.complex64 if single else torch.complex128, device="cuda",
                        generator=gen)
        xs = x.cpu().numpy().astype(np.complex128).reshape(cols, g.d)
        apart, over = torch.full_like(x, float("nan")), x.clone()
        g.matvec_device(x, apart, cols, single=single)
        g.matvec_device(over, over, cols, single=single)
        shifted = torch.zeros((cols + 1) * g.d, dtype=x.dtype, device="cuda")  # outputs one column along
        shifted[:g.d] = x[:g.d]
        g.matvec_device(shifted[:cols * g.d], shifted[g.d:], cols, single=single)
    tol = 1e-13 if prec == "fp64" else 2e-6
    for j in {0, cols - 1}:
        ref = h.hammult(xs[j])
        for y in (apart, over):
            got = y.view(cols, -1)[j].cpu().numpy()
            assert np.max(np.abs(got - ref)) <= tol * np.max(np.abs(ref)), j
    first = shifted.view(cols + 1, -1)
    assert torch.equal(first[0], x[:g.d]) and torch.equal(first[1], apart[:g.d])


def _extended(g, z):
    """H z (M x M, Z[q, p]) in 80-bit arithmetic from the grid's own tables."""
    ld = np.longdouble
    t1, tab, d = np.array(g.kematrix()).astype(ld), np.array(g.tinv()).astype(ld), ld(g.delta)
    one, lab = np.eye(g.nn, dtype=ld), np.arange(g.m)
    k3 = (np.kron(one, np.kron(one, t1)) + np.kron(one, np.kron(t1, one)) + np.kron(t1, np.kron(one, one)))
    ax = (lab % g.nn, lab // g.nn % g.nn, lab // g.nn ** 2)
    vn = -ld(g.charge) / d ** 3 * tab[tuple(a - g.n + g.nn for a in ax)]
    v = vn[:, None] + vn[None, :] + tab[tuple(a[:, None] - a[None, :] + g.nn for a in ax)] / d ** 3
    zr, zi = z.real.astype(ld), z.imag.astype(ld)
    kr, ki, th = zr @ k3 + k3 @ zr, zi @ k3 + k3 @ zi, ld(g.theta)
    c2, s2, c1, s1 = np.cos(2 * th), np.sin(2 * th), np.cos(th), np.sin(th)
    return c2 * kr + s2 * ki + v * (c1 * zr + s1 * zi), c2 * ki - s2 * kr + v * (c1 * zi - s1 * zr)


@pytest.mark.parametrize("n,prec,single,bound", [
    (1, "fp64", False, 2.008e-16), (1, "fp32", True, 7.137e-8), (1, "fp32", False, 7.586e-8),
    (2, "fp64", False, 1.937e-16), (2, "fp32", True, 6.977e-8), (2, "fp32", False, 7.425e-8)])
def test_one_launch_is_as_accurate_as_two(dex, n, prec, single, bound):
    """The 2-norm error over 40 random vectors against 80-bit arithmetic.  The bounds are the
    errors that two launches, a pass an electron with a running sum an axis, had on the same
    vectors."""
    print(f"case: direct error n={n} {prec} complex64={single}", flush=True)
    err = size = 0.0
    with dex.HeliumGrid(n, 0.5, 0.3, precision=prec) as g:
        for seed in range(40):
            rng = np.random.default_rng(seed)
            x = torch.from_numpy(rng.standard_normal(g.d) + 1j * rng.standard_normal(g.d)).cuda()
            x = x.to(torch.complex64) if single else x
            y = torch.empty_like(x)
            g.matvec_device(x, y, 1, single=single)
            z, got = (t.cpu().numpy().astype(np.complex128).reshape(g.m, g.m) for t in (x, y))
            re, im = _extended(g, z)
            err += float(((got.real - re) ** 2 + (got.imag - im) ** 2).sum())
            size += float((re ** 2 + im ** 2).sum())
    print(f"  {(err / size) ** 0.5:.4e}", flush=True)
    assert (err / size) ** 0.5 <= bound
