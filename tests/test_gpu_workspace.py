"""Work vectors kept between calls: calls that share them give what calls on
fresh memory give, from several contexts and threads, and the last context to
close gives the memory back."""
import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dex():
    import doublyexcited_amd as d

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return d


def _block(g, k, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(k, g.m, g.m, dtype=torch.complex128, device="cuda", generator=gen)
    return (0.5 * (x + x.transpose(1, 2))).contiguous().view(-1)


@pytest.mark.parametrize("n,k,order", [(2, 3, 2), (4, 5, 4)])
def test_calls_that_share_work_vectors_agree_with_fresh_ones(dex, n, k, order):
    """Each thread's inner solves on its own context, several at once, are
    bitwise the first (serial) ones: the same kernels on the same inputs."""
    print(f"case: shared work vectors N={n} k={k} order={order}", flush=True)
    with dex.HeliumGrid(n, 0.5, 0.3) as g:
        xs = [_block(g, k, s) for s in range(3)]
        ref = []
        for x in xs:
            y = torch.empty_like(x)
            g.precblock_device(x, y, k, -0.7 - 0.002j, order, symmetry=1)
            ref.append(y)
    bad = []

    def work(i):
        try:
            with dex.HeliumGrid(n, 0.5, 0.3) as h:
                for _ in range(3):
                    y = torch.full_like(xs[i], float("nan"))
                    h.precblock_device(xs[i], y, k, -0.7 - 0.002j, order, symmetry=1)
                    if not torch.equal(y, ref[i]):
                        bad.append(i)
        except Exception as e:  # reported below: an assertion in a thread is lost
            bad.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_the_last_context_gives_the_memory_back(dex):
    print("case: memory given back", flush=True)
    x = None
    with dex.HeliumGrid(4, 0.5, 0.3) as g:
        x = _block(g, 4, 1)
        y = torch.empty_like(x)
        torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    with dex.HeliumGrid(4, 0.5, 0.3) as g:
        g.precblock_device(x, y, 4, -0.7 - 0.002j, 6, symmetry=1)  # 28 vectors of 8.5 MB
        held = before - torch.cuda.mem_get_info()[0]
        assert held >= 28 * 16 * g.d
    assert before - torch.cuda.mem_get_info()[0] <= 32 << 20  # allocator granularity


def test_inner_solve_uses_its_exchange_symmetry(dex):
    """The inner solve of a symmetric block applies H by the exchange-symmetric
    passes, and agrees with the general ones to rounding."""
    print("case: inner solve symmetry", flush=True)
    with dex.HeliumGrid(3, 0.5, 0.3) as g:
        x = _block(g, 3, 7)
        got = {}
        for sym in (0, 1):
            g.reset_kernel_stats()
            y = torch.empty_like(x)
            g.precblock_device(x, y, 3, -0.7 - 0.002j, 3, symmetry=sym)
            totals = g.kernel_totals()
            assert (totals["symadd"][0] > 0) == (sym != 0) and (totals["pass2"][0] > 0) == (sym == 0)
            got[sym] = y
        assert (got[0] - got[1]).abs().max().item() <= 1e-9 * got[0].abs().max().item()


def test_idle_work_vectors_are_given_back_on_request(dex):
    print("case: trim idle", flush=True)
    with dex.HeliumGrid(4, 0.5, 0.3) as g:
        x = _block(g, 4, 1)
        y, z = torch.empty_like(x), torch.empty_like(x)
        g.precblock_device(x, y, 4, -0.7 - 0.002j, 6, symmetry=1)
        vec, held = 16 * g.d, dex.idle_bytes()
        assert held >= 28 * vec and held % vec == 0
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        dex.trim_idle(keep_bytes=held - 3 * vec + 1)  # whole vectors: one byte less than three takes three
        assert dex.idle_bytes() == held - 3 * vec
        dex.trim_idle()
        assert dex.idle_bytes() == 0 and torch.cuda.mem_get_info()[0] - free >= held
        g.precblock_device(x, z, 4, -0.7 - 0.002j, 6, symmetry=1)
        assert torch.equal(y, z) and dex.idle_bytes() == held


def test_server_keeps_idle_work_vectors_under_its_cap(dex):
    """Requests one after the other while another context stays open: each leaves its work
    vectors listed, in sizes (three grids, two formats) that the next cannot use.  The cap
    holds the largest request; the device's use beyond the start stays under it, where all
    that the requests leave would not."""
    from doublyexcited_amd.serve import Request, Server

    print("case: server cap with idle work vectors", flush=True)
    reqs = [Request(arrival=0.0, rid=i, n=n, delta=0.5, theta=0.3, sigma=-0.78 - 0.002j, nev=8, tol=1e-9, maxit=2,
                    seed=i, inner_iter=4, guard=2, precision=p)
            for i, (n, p) in enumerate(((6, "fp64"), (6, "mixed"), (5, "fp64"), (5, "mixed"), (4, "fp64")))]
    need = [r.need() for r in reqs]
    used = []  # bytes after each request

    class Watched(Server):
        def _execute(self, req):
            out = super()._execute(req)
            torch.cuda.empty_cache()
            torch.cuda.synchronize()
            used.append(base - torch.cuda.mem_get_info()[0])
            return out

    with dex.HeliumGrid(1, 0.5, 0.3):
        dex.trim_idle()
        torch.cuda.empty_cache()
        torch.cuda.synchronize()
        base = torch.cuda.mem_get_info()[0]
        cap = max(need)
        out = Watched(hbm_cap_bytes=cap, slots=1).run(reqs, realtime=False)
        assert all(r.ok for r in out), [r.error for r in out]
        print("case: used", used, need, flush=True)
        assert used[0] > 0.5 * need[0] and max(used) <= cap, (used, need)
        dex.trim_idle()
