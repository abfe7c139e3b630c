"""Performance cases of the helium matvec and block-eigensolver path.

Each case is one call, or one short run, of a public entry point of ``HeliumGrid``
as a solve, a request server or a caller of the operator makes it:

  matvec     Y = H X on device columns (``matvec_device``): general vectors
             (symmetry 0) and exchange-(anti)symmetric ones (+1 / -1), complex128
             in FP64 and complex64 in single precision;
  graph      the same through a captured graph (``matvec_graph``), as loops of
             many small solves replay it;
  dots       bras^H kets of two blocks (``dots_device``, MYDOTSUB);
  residuals  ||H x - e x|| / ||x|| of returned pairs (``residuals_device``);
  precblock  the inner solve of order m on a block (``precblock_device``);
  gplmr      iterations of the eigensolver on a block (``gplmr_eig_device``).

The mixed-precision solve has no case of its own: its complex128 eigenvectors
carry the rounding of its single-precision matvecs.  Its matvecs are those of
the complex64 cases.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from doublyexcited_amd import HeliumGrid

SIGMAS = (-0.78, -0.69, -0.60)  # Re sigma of the served requests (au); Im sigma is -0.002
WORK_MOST = 3.8e10              # bytes + flops / 50 of the most expensive drawn case


def listed() -> list[dict]:
    return [
        # the smallest call: one general vector on a 5-point grid, all launch latency
        {"name": "matvec-nn5", "op": "matvec", "nn": 5, "delta": 0.5, "theta": 0.3, "cols": 1, "symmetry": 0,
         "single": False},
        # a block of small vectors replayed as one launch
        {"name": "graph-nn9-singlet", "op": "graph", "nn": 9, "delta": 0.5, "theta": 0.3, "cols": 16,
         "symmetry": 1, "single": False},
        # the search block of the 11-point solve (8 wanted columns and 2 guards)
        {"name": "matvec-nn11-singlet", "op": "matvec", "nn": 11, "delta": 0.5, "theta": 0.3, "cols": 10,
         "symmetry": 1, "single": False},
        # general vectors, as a caller of the operator without exchange symmetry has them
        {"name": "matvec-nn13-general", "op": "matvec", "nn": 13, "delta": 0.47, "theta": 0.25, "cols": 3,
         "symmetry": 0, "single": False},
        # complex64 search-block columns of a mixed-precision triplet solve
        {"name": "matvec-nn19-triplet-c64", "op": "matvec", "nn": 19, "delta": 0.42, "theta": 0.3, "cols": 4,
         "symmetry": -1, "single": True},
        # the largest grid of the served stream: a group of four columns in FP64
        {"name": "matvec-nn21-singlet", "op": "matvec", "nn": 21, "delta": 0.4, "theta": 0.35, "cols": 4,
         "symmetry": 1, "single": False},
        # the largest grid built, FP64 (the mixed solve's AX there)
        {"name": "matvec-nn25-general", "op": "matvec", "nn": 25, "delta": 0.35, "theta": 0.3, "cols": 1,
         "symmetry": 0, "single": False},
        # a projection of one block against a wider basis
        {"name": "dots-nn15", "op": "dots", "nn": 15, "delta": 0.45, "theta": 0.3, "cols": 12, "kets": 10},
        # the check of a served request's eight returned pairs
        {"name": "residuals-nn17", "op": "residuals", "nn": 17, "delta": 0.5, "theta": 0.4, "cols": 8},
        # the whole-block inner solve of a small served request (4 wanted columns and 2 guards, order 8)
        {"name": "precblock-nn13", "op": "precblock", "nn": 13, "delta": 0.47, "theta": 0.3, "cols": 6,
         "symmetry": 1, "order": 8, "sigma": -0.69},
        # one four-column group of the inner solve on the largest served grid, order 4
        {"name": "precblock-nn21", "op": "precblock", "nn": 21, "delta": 0.4, "theta": 0.35, "cols": 4,
         "symmetry": 1, "order": 4, "sigma": -0.78},
        # the eigensolver's first iterations on the 11-point grid: 8 pairs and 2 guard columns
        {"name": "gplmr-nn11", "op": "gplmr", "nn": 11, "delta": 0.5, "theta": 0.3, "cols": 8, "guard": 2,
         "symmetry": 1, "order": 8, "ns": 4, "iters": 2, "sigma": -0.78},
    ]


def _odd(rng, lo: int, hi: int) -> int:
    """An odd grid size whose vector length, NN^6, is spread over its logarithm."""
    x = math.exp(rng.uniform(math.log(lo - 1), math.log(hi + 1)))
    return max(lo, min(hi, 2 * int(x / 2) + 1))


def draw(rng) -> dict:
    while True:
        op = rng.choice(("matvec", "matvec", "matvec", "matvec", "graph", "dots", "residuals", "precblock",
                         "precblock", "gplmr"))
        case = {"op": op, "delta": round(rng.uniform(0.35, 0.6), 4), "theta": round(rng.uniform(0.2, 0.5), 4)}
        if op == "matvec":
            single = rng.random() < 0.35
            sym = rng.choice((0, 1, 1, -1))
            hi = 25 if single or sym == 0 else 21
            case |= {"nn": _odd(rng, 5, hi), "cols": rng.randint(1, 16), "symmetry": sym, "single": single}
        elif op == "graph":
            case |= {"nn": _odd(rng, 5, 11), "cols": rng.randint(1, 16), "symmetry": rng.choice((0, 1, -1)),
                     "single": False}
        elif op == "dots":
            case |= {"nn": _odd(rng, 9, 19), "cols": rng.randint(1, 24), "kets": rng.randint(1, 24)}
        elif op == "residuals":
            case |= {"nn": _odd(rng, 9, 21), "cols": rng.choice((4, 8, 16))}
        elif op == "precblock":
            case |= {"nn": _odd(rng, 9, 21), "cols": rng.randint(2, 10), "symmetry": rng.choice((1, 1, -1, 0)),
                     "order": rng.randint(2, 8), "sigma": rng.choice(SIGMAS)}
        else:
            case |= {"nn": _odd(rng, 7, 13), "cols": rng.choice((4, 8)), "guard": 2, "symmetry": 1,
                     "order": rng.choice((4, 8)), "ns": rng.choice((1, 4)), "iters": 2,
                     "sigma": rng.choice(SIGMAS)}
        w = work(case)
        columns = case["cols"] + case.get("kets", case["cols"])
        if w["bytes"] + w["flops"] / 50 <= WORK_MOST and columns * 16 * case["nn"] ** 6 <= 13e9:
            return case


# ---- inputs ---------------------------------------------------------------------

def _block(nn: int, cols: int, symmetry: int, single: bool, gen) -> torch.Tensor:
    """Complex Gaussian columns, exchange-(anti)symmetric for symmetry +1 / -1."""
    m = nn ** 3
    dtype = torch.complex64 if single else torch.complex128
    x = torch.empty(cols, m, m, dtype=dtype, device="cuda")
    for c in range(cols):
        v = torch.randn(m, m, dtype=dtype, device="cuda", generator=gen)
        x[c] = 0.5 * (v + symmetry * v.T) if symmetry else v
    return x.reshape(-1)


def _generator(seed: int):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _sigma(case: dict) -> complex:
    return complex(case["sigma"], -0.002)


def prepare(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    op, nn, cols = case["op"], case["nn"], case["cols"]
    single = bool(case.get("single", False))
    grid = HeliumGrid(nn // 2, case["delta"], case["theta"], precision="fp32" if single else "fp64")
    state = {"case": case, "grid": grid}
    state["x"] = _block(nn, cols, case.get("symmetry", 0), single, gen)
    if op in ("matvec", "graph", "precblock"):
        state["y"] = torch.empty_like(state["x"])
    if op == "graph":
        state["graph"] = grid.matvec_graph(state["x"], state["y"], symmetry=case["symmetry"], single=single)
    elif op == "dots":
        state["kets"] = _block(nn, case["kets"], 0, False, gen)
    elif op == "residuals":
        state["e"] = _energies(cols, seed)
    elif op == "gplmr":
        state["work"] = torch.empty_like(state["x"])
    return state


def _energies(cols: int, seed: int) -> np.ndarray:
    r = np.random.default_rng(seed)
    return -0.8 + 0.5 * r.random(cols) - 0.3j * r.random(cols)


def run(state: dict):
    case, grid = state["case"], state["grid"]
    op = case["op"]
    if op == "matvec":
        grid.matvec_device(state["x"], state["y"], single=case["single"], symmetry=case["symmetry"])
        return state["y"]
    if op == "graph":
        state["graph"].launch()
        grid.sync()
        return state["y"]
    if op == "dots":
        return grid.dots_device(state["x"], state["kets"], case["cols"], case["kets"])
    if op == "residuals":
        return grid.residuals_device(state["x"], state["e"])
    if op == "precblock":
        grid.precblock_device(state["x"], state["y"], case["cols"], _sigma(case), case["order"], case["symmetry"])
        return state["y"]
    # the solver overwrites its start block
    state["work"].copy_(state["x"])
    r = grid.gplmr_eig_device(state["work"], _sigma(case), case["cols"], ns=case["ns"], maxit=case["iters"],
                              tol=1e-10, inner_iter=case["order"], symmetry=case["symmetry"], guard=case["guard"])
    # an eigenvector's phase is arbitrary: fixed by its product with the block's first start column
    x = state["work"].view(case["cols"], -1)
    p = x @ state["x"].view(case["cols"], -1)[0].conj()
    x *= (p.conj() / p.abs())[:, None]
    return {"x": state["work"], "e": r.e, "max_residual": r.max_residual}


# ---- work -----------------------------------------------------------------------

def _inner_flops(nn: int, cols: int, order: int, symmetry: int) -> float:
    """The inner solve on `cols` columns: the matvecs, and a Gram and a combination of each new block
    against the basis so far, 8 flops a complex multiply-add."""
    d = float(nn) ** 6
    blocks = sum(range(1, order + 2))
    return order * cols * _matvec_flops(nn, symmetry) + 8.0 * d * cols * cols * (2 * blocks + order)


def _matvec_flops(nn: int, symmetry: int) -> float:
    """Six axes of NN real-by-complex multiply-adds an entry (three with exchange symmetry) and the potential."""
    return ((12.0 if symmetry else 24.0) * nn + 14.0) * float(nn) ** 6


def work(case: dict) -> dict:
    op, nn, cols = case["op"], case["nn"], case["cols"]
    d = float(nn) ** 6
    sym = case.get("symmetry", 0)
    entry = 8.0 if case.get("single") else 16.0
    if op in ("matvec", "graph"):
        return {"bytes": 2 * entry * cols * d, "flops": cols * _matvec_flops(nn, sym)}
    if op == "dots":
        return {"bytes": entry * (cols + case["kets"]) * d, "flops": 8.0 * d * cols * case["kets"]}
    if op == "residuals":
        return {"bytes": entry * cols * d, "flops": cols * (_matvec_flops(nn, 0) + 12.0 * d)}
    if op == "precblock":
        return {"bytes": 2 * entry * cols * d, "flops": _inner_flops(nn, cols, case["order"], sym)}
    block, ns = cols + case["guard"], case["ns"]
    basis = (3 + ns) * block
    each = ((1 + ns) * (_inner_flops(nn, block, case["order"], sym) + block * _matvec_flops(nn, sym))
            + 8.0 * d * (1.5 * basis * basis + 2 * basis * 2 * block))
    return {"bytes": 2 * entry * cols * d, "flops": block * _matvec_flops(nn, sym) + case["iters"] * each}


# ---- the same in plain 64-bit arithmetic ----------------------------------------------

@functools.lru_cache(maxsize=4)
def _coulomb_table(delta: float, half: int = 22, factor: int = 4) -> np.ndarray:
    """Regularised 1/r of the sinc grid at labels -51..51 per axis: the bare delta^3/r, corrected
    on the small grid so that the kinetic operator applied to it is 2 pi at the origin."""
    big = half * factor

    def kinetic(a, b):
        k = a[:, None] - b[None, :]
        with np.errstate(divide="ignore"):
            off = np.where(k % 2 == 0, 1.0, -1.0) / (k.astype(float) ** 2)
        return np.where(k == 0, np.pi ** 2 / 6, off) / delta ** 2

    labels, small = np.arange(-big, big + 1), np.arange(-half, half + 1)
    s = slice(big - half, big + half + 1)

    def bare(a, b, c):
        r = np.sqrt((a.astype(float) ** 2)[:, None, None] + (b.astype(float) ** 2)[None, :, None]
                    + (c.astype(float) ** 2)[None, None, :])
        with np.errstate(divide="ignore"):
            return np.where(r == 0, 0.0, delta ** 2 / r)

    line = np.tensordot(kinetic(small, labels), bare(labels, small, small), axes=(1, 0))  # [i, j, k]
    rhs = -(line + line.transpose(1, 0, 2) + line.transpose(1, 2, 0))
    rhs[half, half, half] += 2 * np.pi
    w, v = np.linalg.eigh(kinetic(small, small))
    q = np.einsum("ai,bj,ck,abc->ijk", v, v, v, rhs, optimize=True)
    q /= w[:, None, None] + w[None, :, None] + w[None, None, :]
    q = np.einsum("ia,jb,kc,abc->ijk", v, v, v, q, optimize=True)
    out_labels = np.arange(-51, 52)
    table = bare(out_labels, out_labels, out_labels)
    c = slice(51 - half, 51 + half + 1)
    table[c, c, c] += q
    return table


class _Exact:
    """H as dense M x M factors: Y = s2 (X K + K X) + c1 V o X on X[q, p]."""

    def __init__(self, nn: int, delta: float, theta: float):
        m = nn ** 3
        table = torch.from_numpy(_coulomb_table(delta)).cuda()
        lab = torch.arange(m, device="cuda")
        i, j, k = lab % nn, lab // nn % nn, lab // nn ** 2
        h = nn // 2
        nuc = -2.0 / delta ** 3 * table[51 + i - h, 51 + j - h, 51 + k - h]
        at = [51 + a[:, None] - a[None, :] for a in (i, j, k)]
        self.v = nuc[:, None] + nuc[None, :] + table[at[0], at[1], at[2]] / delta ** 3
        a = torch.arange(nn, device="cuda")
        d = a[:, None] - a[None, :]
        t = torch.where(d == 0, math.pi ** 2 / 6, (1.0 - 2.0 * (d % 2)) / d.double() ** 2)
        one = torch.eye(nn, dtype=torch.float64, device="cuda")
        self.k = (torch.kron(one, torch.kron(one, t)) + torch.kron(one, torch.kron(t, one))
                  + torch.kron(t, torch.kron(one, one)))
        self.s2 = complex(math.cos(2 * theta), -math.sin(2 * theta)) / delta ** 2
        self.c1 = complex(math.cos(theta), -math.sin(theta))
        self.m = m

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        """One flat vector; two real products a part."""
        z = x.reshape(self.m, self.m).to(torch.complex128)
        parts = []
        for r in (z.real.contiguous(), z.imag.contiguous()):
            parts.append(r @ self.k + self.k @ r)
        y = torch.complex(*parts)
        y *= self.s2
        return (y + self.c1 * (self.v * z)).reshape(-1)


def _columns(x: torch.Tensor, cols: int) -> torch.Tensor:
    return x.view(cols, -1)


def _gram(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """a^H b of two blocks whose columns are the rows of a and b."""
    return torch.stack([(v.conj() * b).sum(1) for v in a])


def _exact_inner(h: _Exact, b: torch.Tensor, order: int, sigma: complex) -> torch.Tensor:
    """argmin ||(H - sigma) x - b|| over the block Krylov space of H and b (columns as rows of b)."""
    cols = b.shape[0]

    def orthonormal(q, w):  # rows of w against the rows of q and each other, three times over
        for _ in range(3):
            if q is not None:
                w = w - _gram(q, w).T @ q
            g = torch.linalg.cholesky(_gram(w, w).conj())  # rows: w_i w_j^H
            w = torch.linalg.inv(g) @ w
        return w

    q = orthonormal(None, b)
    images = []
    for step in range(order):
        last = q[-cols:]
        image = torch.stack([h(v) - sigma * v for v in last])
        images.append(image)
        if step + 1 < order:
            q = torch.cat([q, orthonormal(q, image)])
    a = torch.cat(images)
    basis = orthonormal(None, a)  # least squares through an orthonormal basis of the images
    y = torch.linalg.solve(_gram(basis, a), _gram(basis, b))
    return y.T @ q


def exact(case: dict, seed: int):
    op, nn, cols = case["op"], case["nn"], case["cols"]
    if op == "gplmr":
        return None
    gen = _generator(seed)
    x = _block(nn, cols, case.get("symmetry", 0), bool(case.get("single", False)), gen)
    if op == "dots":
        kets = _block(nn, case["kets"], 0, False, gen)
        return _gram(_columns(x, cols), _columns(kets, case["kets"])).cpu().numpy()
    h = _Exact(nn, case["delta"], case["theta"])
    xc = _columns(x, cols)
    if op in ("matvec", "graph"):
        return torch.cat([h(v) for v in xc])
    if op == "residuals":
        e = _energies(cols, seed)
        return np.array([float(torch.linalg.vector_norm(h(v) - complex(z) * v) / torch.linalg.vector_norm(v))
                         for v, z in zip(xc, e)])
    if cols * (2 * case["order"] + 3) * 16 * nn ** 6 > 120e9:
        return None
    return _exact_inner(h, xc, case["order"], _sigma(case)).reshape(-1)
