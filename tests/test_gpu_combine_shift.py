"""The block combinations on shifted columns, out_j = sum_i (a_i - sigma_i b_i) C(i, j):
the difference is formed in FP64 also where a and b are complex64, as the Arnoldi blocks
(H - sigma) Q of a single-precision inner solve are.

Every kernel: registers for 4, 8, 12, 16 and 48 outputs, LDS for 17 to 32, tiles of
exchange-(anti)symmetric columns for 4 to 16; odd lengths and ragged tiles.  Bound: FP64
sums of at most 9 products and their differences, 1e-14 of the largest sum of moduli (an
FP32 difference at |sigma| ~ 1000 would be off by 1e-8 of it)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DESC = np.dtype([("a", "u8"), ("b", "u8"), ("sre", "f8"), ("sim", "f8"), ("bslot", "i4"), ("fmt", "i4")])


@pytest.fixture(scope="module")
def kernels():
    from doublyexcited_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib = _lib.load()
    p, i, l, b = C.c_void_p, C.c_int, C.c_int64, C.c_bool
    rows = lib["_ZN3dex14launch_combineEPKNS_7ColDescEiiPKNS_4Dbl2ES5_lbP12ihipStream_t"]
    rows.argtypes = [p, i, i, p, p, l, b, p]
    halves = lib["_ZN3dex18launch_combine_symEPKNS_7ColDescEiiPKNS_4Dbl2ES5_iibP12ihipStream_t"]
    halves.argtypes = [p, i, i, p, p, i, i, b, p]
    ld = lib["_ZN3dex10combine_ldEi"]
    ld.argtypes = [i]
    return rows, halves, ld


@pytest.mark.parametrize("m,sign,nout", [
    (0, 0, 1), (0, 0, 4), (0, 0, 7), (0, 0, 12), (0, 0, 16), (0, 0, 17), (0, 0, 32), (0, 0, 33), (0, 0, 48),
    (45, 1, 1), (45, -1, 4), (33, 1, 8), (45, -1, 11), (64, 1, 16)])
@pytest.mark.parametrize("single", [True, False])
def test_combination_of_shifted_columns(kernels, m, sign, nout, single):
    print(f"case: shifted columns m={m} sign={sign} nout={nout} complex64={single}", flush=True)
    rows, halves, ld = kernels
    d = m * m if m else 1003
    dtype = torch.complex64 if single else torch.complex128
    gen = torch.Generator(device="cuda").manual_seed(nout + m)

    def column(kind):
        v = torch.randn(d, dtype=kind, device="cuda", generator=gen)
        return (0.5 * (v.view(m, m) + sign * v.view(m, m).T)).contiguous().view(-1) if m else v

    # three shifted columns, one alone in each format
    a = [column(dtype) for _ in range(4)] + [column(torch.complex128)]
    b = [column(dtype) for _ in range(3)] + [None, None]
    sig = [900.0 - 400.0j, -0.7 - 0.002j, 0.3j, 0.0, 0.0]
    out = [torch.full((d,), float("nan"), dtype=torch.complex128, device="cuda") for _ in range(nout)]
    desc = np.zeros(5 + nout, DESC)
    for k in range(5):
        desc[k] = (a[k].data_ptr(), 0 if b[k] is None else b[k].data_ptr(), sig[k].real, sig[k].imag, -1,
                   int(a[k].dtype == torch.complex64))
    for k in range(nout):
        desc[5 + k] = (out[k].data_ptr(), 0, 0.0, 0.0, -1, 0)
    cm = torch.randn(5, nout, dtype=torch.complex128, device="cuda", generator=gen)
    padded = torch.zeros(5, ld(nout), dtype=torch.complex128, device="cuda")
    padded[:, :nout] = cm
    descs = torch.from_numpy(desc.view(np.uint8).copy()).cuda()
    torch.cuda.synchronize()
    if m:
        st = halves(descs.data_ptr(), 5, nout, padded.data_ptr(), None, m, sign, False, None)
    else:
        st = rows(descs.data_ptr(), 5, nout, padded.data_ptr(), None, d, False, None)
    torch.cuda.synchronize()
    assert st == 0
    terms = [[a[k].to(torch.complex128)] + ([] if b[k] is None else [-sig[k] * b[k].to(torch.complex128)])
             for k in range(5)]
    for j in range(nout):
        ref = sum(cm[k, j] * t for k in range(5) for t in terms[k])
        size = sum(cm[k, j].abs() * t.abs() for k in range(5) for t in terms[k]).max().item()
        assert (out[j] - ref).abs().max().item() <= 1e-14 * size, j
