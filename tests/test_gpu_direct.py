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
