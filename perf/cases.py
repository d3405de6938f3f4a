"""The workloads whose speed this library is held to.

Each case is one pass through ``numax_amd.linalg``'s public functions as a
user's program calls them: dense solves from the smallest order to the
benchmark's, Cholesky, least squares, the mixed-precision solve with one and
many right-hand sides, and the batched solvers.  Sizes are the repository's
own benchmark and test sizes, or generic ones beside them.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes the inputs on the GPU, ``run`` is one pass, ``work`` the
bytes and operations the pass cannot do without, ``exact`` the same results
in 64 bits from torch alone.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from numax_amd import linalg as nl

DEVICE = "cuda:0"
DTYPES = {"f64": torch.float64, "f32": torch.float32}


def listed() -> list:
    return [
        # the smallest dense call: one small system, where launches count
        {"name": "solve_f64_n100", "kind": "solve", "dtype": "f64", "n": 100, "nrhs": 1, "tuned": False},
        # an ordinary system with the functions' own defaults
        {"name": "solve_f64_n1000", "kind": "solve", "dtype": "f64", "n": 1000, "nrhs": 1, "tuned": False},
        # the benchmark's plain FP64 factor + solve: a large matrix at the
        # panel widths lu_factor's docstring recommends for it, factor kept
        {"name": "lu_f64_n8192_rhs16", "kind": "lu", "dtype": "f64", "n": 8192, "nrhs": 16, "tuned": True},
        # the benchmark's FP64 Cholesky factor + solve
        {"name": "chol_f64_n8192_rhs16", "kind": "cholesky", "dtype": "f64", "n": 8192, "nrhs": 16, "tuned": True},
        # an ordinary covariance solve in single precision, odd order, defaults
        {"name": "chol_f32_n1301", "kind": "cholesky", "dtype": "f32", "n": 1301, "nrhs": 1, "tuned": False},
        # a regression: tall least squares in numax's device precision, defaults
        {"name": "lstsq_f32_2500x300", "kind": "lstsq", "dtype": "f32", "m": 2500, "n": 300, "nrhs": 1},
        # the headline: mixed-precision LU with refinement to FP64 accuracy
        {"name": "mpir_n16384", "kind": "mpir", "n": 16384, "nrhs": 1},
        # the same solver at a smaller, ragged order with a block of right-hand sides
        {"name": "mpir_n5000_rhs64", "kind": "mpir", "n": 5000, "nrhs": 64},
        # the benchmark's batch of uneven systems, half LU and half Cholesky
        {"name": "batched_20000", "kind": "batched", "count": 20000},
        # the benchmark's batch of small symmetric eigenproblems
        {"name": "eigh_65536", "kind": "eigh", "count": 65536},
        # the benchmark's batch of tall-skinny regressions
        {"name": "lstsq_batched_4096", "kind": "lstsq_batched", "count": 4096, "m": 1024, "n": 32},
        # map_blocks over many small dense systems in its structure-of-arrays layout
        {"name": "map_blocks_f64_n24", "kind": "map_blocks", "dtype": "f64", "step": "lu", "n": 24, "batch": 100000},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["solve", "solve", "lu", "cholesky", "cholesky", "lstsq", "mpir", "batched", "eigh",
                       "lstsq_batched", "map_blocks"])
    if kind in ("solve", "lu"):
        n = _log_int(rng, 48, 1500) if kind == "solve" else _log_int(rng, 1500, 8192)
        return {"kind": kind, "dtype": rng.choice(["f64", "f64", "f32"]), "n": n, "nrhs": _log_int(rng, 1, 64),
                "tuned": n > 1500}
    if kind == "cholesky":
        n = _log_int(rng, 48, 8192)
        return {"kind": kind, "dtype": rng.choice(["f64", "f32"]), "n": n, "nrhs": _log_int(rng, 1, 64),
                "tuned": n > 1500}
    if kind == "lstsq":
        n = _log_int(rng, 8, 600)
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "m": int(n * rng.uniform(2.0, 10.0)), "n": n,
                "nrhs": _log_int(rng, 1, 16)}
    if kind == "mpir":
        return {"kind": kind, "n": _log_int(rng, 1000, 12000), "nrhs": rng.choice([1, 1, _log_int(rng, 2, 64)])}
    if kind == "batched":
        return {"kind": kind, "count": _log_int(rng, 64, 20000)}
    if kind == "eigh":
        return {"kind": kind, "count": _log_int(rng, 256, 65536)}
    if kind == "lstsq_batched":
        n = rng.randint(2, 32)
        return {"kind": kind, "count": _log_int(rng, 32, 4096), "m": _log_int(rng, 2 * n, 2000), "n": n}
    n = _log_int(rng, 2, 64)
    return {"kind": "map_blocks", "dtype": rng.choice(["f64", "f32"]), "step": rng.choice(["lu", "cholesky"]), "n": n,
            "batch": max(1000, min(1000000, _log_int(rng, 20_000_000, 80_000_000) // (n * n)))}


# ---- inputs ------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float64):
    return torch.randn(shape, dtype=dtype, device=DEVICE, generator=g)


def _spd(g, n: int):
    """A covariance-like matrix: G G^T / n + I."""
    m = _randn(g, n, n)
    return (m @ m.T / n + torch.eye(n, dtype=torch.float64, device=DEVICE)).contiguous()


def _batch_layout(count: int):
    """The uneven batch's orders (8..256), kinds (LU and Cholesky in turn) and offsets."""
    r = random.Random(count)
    n = np.array([r.randint(8, 256) for _ in range(count)], dtype=np.int32)
    kind = (np.arange(count) % 2).astype(np.uint8)
    offa = np.zeros(count, dtype=np.int64)
    offb = np.zeros(count, dtype=np.int64)
    offa[1:] = np.cumsum(n.astype(np.int64) ** 2)[:-1]
    offb[1:] = np.cumsum(n.astype(np.int64))[:-1]
    return n, kind, offa, offb


def _scatter(dst, blocks, offsets):
    """Writes blocks[i] (equal shapes) at element offset offsets[i] of dst."""
    each = blocks[0].numel()
    at = torch.as_tensor(offsets, device=DEVICE)[:, None] + torch.arange(each, device=DEVICE)
    dst[at.reshape(-1)] = blocks.reshape(-1)


def _batched_inputs(count: int, seed: int):
    n, kind, offa, offb = _batch_layout(count)
    g = _gen(seed)
    a = torch.empty(int((n.astype(np.int64) ** 2).sum()), dtype=torch.float64, device=DEVICE)
    for size in np.unique(n):
        size = int(size)
        eye = torch.eye(size, dtype=torch.float64, device=DEVICE)
        idx = np.flatnonzero((n == size) & (kind == 0))
        if idx.size:
            m = torch.rand((idx.size, size, size), dtype=torch.float64, device=DEVICE, generator=g) * 2 - 1
            _scatter(a, m + 0.1 * size * eye, offa[idx])
        idx = np.flatnonzero((n == size) & (kind == 1))
        if idx.size:
            m = _randn(g, idx.size, size, size)
            _scatter(a, torch.bmm(m, m.transpose(1, 2).contiguous()) / size + eye, offa[idx])
    return a, _randn(g, int(n.sum())), n, kind, offa, offb


EIGH_SIZES = (24, 32, 48, 64)


def _eigh_layout(count: int):
    n = np.sort(np.resize(np.array(EIGH_SIZES, dtype=np.int32), count))
    offa = np.zeros(count, dtype=np.int64)
    offw = np.zeros(count, dtype=np.int64)
    offa[1:] = np.cumsum(n.astype(np.int64) ** 2)[:-1]
    offw[1:] = np.cumsum(n.astype(np.int64))[:-1]
    return n, offa, offw


def _eigh_inputs(count: int, seed: int):
    """Of each order half finite-difference Hamiltonians of a harmonic well,
    half symmetrized Gaussian matrices."""
    n, offa, offw = _eigh_layout(count)
    g = _gen(seed)
    a = torch.empty(int((n.astype(np.int64) ** 2).sum()), dtype=torch.float32, device=DEVICE)
    for size in EIGH_SIZES:
        idx = np.flatnonzero(n == size)
        half = idx.size // 2
        m = _randn(g, idx.size, size, size)
        m = 0.5 * (m + m.transpose(1, 2))
        if half:
            h = 8.0 / (size - 1)
            x = torch.linspace(-4.0, 4.0, size, dtype=torch.float64, device=DEVICE)
            omega = 0.5 + 1.5 * torch.rand(half, 1, dtype=torch.float64, device=DEVICE, generator=g)
            off = torch.full((size - 1,), -0.5 / h ** 2, dtype=torch.float64, device=DEVICE)
            m[:half] = torch.diag(off, 1) + torch.diag(off, -1)
            m[:half] += torch.diag_embed(1.0 / h ** 2 + 0.5 * omega ** 2 * x ** 2)
        if idx.size:
            _scatter(a, m.to(torch.float32), offa[idx])
    return a, n, offa, offw


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    g = _gen(seed)
    st = {"case": case}
    dt = DTYPES[case.get("dtype", "f64")]
    if kind in ("solve", "lu", "mpir"):
        n = case["n"]
        a = _randn(g, n, n)
        if dt is torch.float32:
            # single precision: a well-conditioned system, as one would trust to it
            a = torch.rand((n, n), dtype=torch.float64, device=DEVICE, generator=g) * 2 - 1
            a += 0.1 * n * torch.eye(n, dtype=torch.float64, device=DEVICE)
        st["a"] = a.to(dt)
        st["b"] = (_randn(g, n) if case["nrhs"] == 1 else _randn(g, n, case["nrhs"])).to(dt)
    elif kind == "cholesky":
        n = case["n"]
        st["a"] = _spd(g, n).to(dt)
        st["b"] = (_randn(g, n) if case["nrhs"] == 1 else _randn(g, n, case["nrhs"])).to(dt)
    elif kind == "lstsq":
        st["a"] = _randn(g, case["m"], case["n"]).to(dt)
        st["b"] = (_randn(g, case["m"]) if case["nrhs"] == 1 else _randn(g, case["m"], case["nrhs"])).to(dt)
    elif kind == "batched":
        st["a"], st["b"], st["n"], st["kinds"], st["offa"], st["offb"] = _batched_inputs(case["count"], seed)
    elif kind == "eigh":
        st["a"], st["n"], st["offa"], st["offw"] = _eigh_inputs(case["count"], seed)
    elif kind == "lstsq_batched":
        st["a"] = _randn(g, case["count"], case["m"], case["n"], dtype=torch.float32)
        st["b"] = _randn(g, case["count"], case["m"], dtype=torch.float32)
    else:
        n, batch = case["n"], case["batch"]
        xs = torch.empty((n * n + n, batch), dtype=dt, device=DEVICE)
        xs.uniform_(-1.0, 1.0, generator=g)
        mats = xs[:n * n].view(n, n, batch)
        if case["step"] == "cholesky":
            mats.copy_(0.5 * (mats + mats.transpose(0, 1)))
        # diagonally dominant, so every step kind has a well-posed problem
        mats.diagonal(dim1=0, dim2=1).add_(float(n))
        st["xs"] = xs
    return st


# ---- one pass ------------------------------------------------------------------

def run(state: dict):
    c = state["case"]
    kind = c["kind"]
    if kind == "solve":
        return nl.solve(state["a"], state["b"])
    if kind == "lu":
        f = nl.lu_factor(state["a"], block=256, base=32)
        return f.factored, f.pivots, f.solve(state["b"])
    if kind == "cholesky":
        low = nl.cholesky(state["a"], block=256) if c["tuned"] else nl.cholesky(state["a"])
        return low, nl.cholesky_solve(low, state["b"])
    if kind == "lstsq":
        return nl.lstsq(state["a"], state["b"])
    if kind == "mpir":
        x, _ = nl.solve_mpir(state["a"], state["b"])
        return x
    if kind == "batched":
        # the step counts follow the rounding of an FP32 factor and are no result of the solve
        r = nl.batched_solve(state["a"], state["b"], state["n"], state["kinds"], state["offa"], state["offb"])
        return r.x, r.info
    if kind == "eigh":
        return nl.eigh_batched(state["a"], state["n"], state["offa"], state["offw"])
    if kind == "lstsq_batched":
        return nl.lstsq_batched(state["a"], state["b"])
    return nl.map_blocks_solve(state["xs"], c["n"], c["step"])


# ---- what a pass cannot do without -----------------------------------------------

def work(case: dict) -> dict:
    kind = case["kind"]
    size = 4 if case.get("dtype") == "f32" else 8
    if kind in ("solve", "lu", "cholesky", "mpir"):
        n, k = case["n"], case["nrhs"]
        factor = n ** 3 / 3 if kind == "cholesky" else 2 * n ** 3 / 3
        kept = n * n if kind in ("lu", "cholesky") else 0
        return {"bytes": size * (n * n + kept + 2 * n * k), "flops": factor + 2 * n * n * k}
    if kind == "lstsq":
        m, n, k = case["m"], case["n"], case["nrhs"]
        return {"bytes": size * (m * n + m * k + n * k), "flops": 2 * n * n * (m - n / 3) + 4 * m * n * k}
    if kind == "batched":
        n = _batch_layout(case["count"])[0].astype(np.float64)
        lu = np.arange(case["count"]) % 2 == 0
        return {"bytes": float((8 * n * n + 16 * n).sum()),
                "flops": float((np.where(lu, 2.0, 1.0) * n ** 3 / 3 + 2 * n * n).sum())}
    if kind == "eigh":
        # about nine n^3 for a symmetric matrix's values and vectors
        n = _eigh_layout(case["count"])[0].astype(np.float64)
        return {"bytes": float((4 * (2 * n * n + n)).sum()), "flops": float((9 * n ** 3).sum())}
    if kind == "lstsq_batched":
        p, m, n = case["count"], case["m"], case["n"]
        return {"bytes": 4 * p * (m * n + m + n), "flops": p * (2 * n * n * (m - n / 3) + 4 * m * n)}
    n, p = case["n"], case["batch"]
    factor = (2 if case["step"] == "lu" else 1) * n ** 3 / 3
    return {"bytes": size * p * (n * n + 2 * n), "flops": p * (factor + 2 * n * n)}


# ---- the same results in 64 bits ----------------------------------------------------

def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "eigh":
        return None  # the order of the values and the vectors' signs are the algorithm's own
    st = prepare(case, seed)
    if kind in ("solve", "mpir", "lu"):
        a, b = st["a"].double(), st["b"].double()
        x = torch.linalg.solve(a, b)
        return x if kind != "lu" else (None, None, x)
    if kind == "cholesky":
        low = torch.linalg.cholesky(st["a"].double())
        b = st["b"].double()
        x = torch.cholesky_solve(b[:, None] if b.dim() == 1 else b, low)
        return low, x[:, 0] if b.dim() == 1 else x
    if kind in ("lstsq", "lstsq_batched"):
        # the normal equations in 64 bits: these matrices are well conditioned
        a, b = st["a"].double(), st["b"].double()
        at = a.transpose(-2, -1).contiguous()
        rhs = b[..., None] if b.dim() == a.dim() - 1 else b
        x = torch.linalg.solve(at @ a, at @ rhs)
        return x[..., 0] if b.dim() == a.dim() - 1 else x
    if kind == "batched":
        x = torch.empty_like(st["b"])
        for size in np.unique(st["n"]):
            idx = np.flatnonzero(st["n"] == size)
            size = int(size)
            at = torch.as_tensor(st["offa"][idx], device=DEVICE)[:, None] + torch.arange(size * size, device=DEVICE)
            bt = torch.as_tensor(st["offb"][idx], device=DEVICE)[:, None] + torch.arange(size, device=DEVICE)
            sol = torch.linalg.solve(st["a"][at].view(-1, size, size), st["b"][bt])
            x[bt.reshape(-1)] = sol.reshape(-1)
        return x, None
    n = case["n"]
    xs = st["xs"].double()
    a = xs[:n * n].t().reshape(-1, n, n).contiguous()
    return torch.linalg.solve(a, xs[n * n:].t().contiguous()).t().contiguous()
