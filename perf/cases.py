"""The calls whose time counts, as a user's program makes them.

Each case is one public entry point on device-resident operands: row-wise
SpGEMM, the outer-product SpGEMM (also in its transposed-output form, where
the operands swap places), MTTKRP, TTM, the CSR transpose and the request
loop of batched SpGEMM.  A program keeps one context (and, when it serves,
its engines) for its whole life, so they are kept here too; inputs are made
on the GPU by torch and handed over as device pointers, and the results come
back as torch views of the arrays the entry point returned.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from sparsews_amd import autotune, serve
from sparsews_amd._lib import check, lib
from sparsews_amd.device import (Context, DeviceArray, DeviceCSF, DeviceCSR, DeviceDCSR, mttkrp, spgemm_outer,
                                 spgemm_rowwise, ttm)

DEV = "cuda"


def listed():
    return [
        # the smallest call: one small product in a longer program, all latency
        {"name": "rowwise_511", "op": "rowwise", "m": 511, "k": 389, "n": 643, "rows": "uniform", "lo": 6, "hi": 6},
        # the row-wise benchmark: short rows only
        {"name": "rowwise_10k_8", "op": "rowwise", "m": 10_000, "k": 10_000, "n": 10_000, "rows": "uniform",
         "lo": 8, "hi": 8},
        # a graph-like product: row lengths from 1 to thousands in one call
        {"name": "rowwise_powerlaw_20k", "op": "rowwise", "m": 20_011, "k": 20_011, "n": 20_011, "rows": "powerlaw",
         "lo": 1, "hi": 4096},
        # the largest request of the serving mix: every row mid-sized
        {"name": "rowwise_uniform_65k", "op": "rowwise", "m": 65_536, "k": 65_536, "n": 65_536, "rows": "uniform",
         "lo": 2, "hi": 64},
        # a small transposed-output product (CSC operand, dense outer level)
        {"name": "outer_2k_8", "op": "outer", "m": 2_003, "k": 1_999, "n": 2_501, "rows": "uniform", "lo": 8, "hi": 8},
        # B^T B of a power-law matrix, the outer-product benchmark at the size
        # that leaves room for several results
        {"name": "outer_powerlaw_80k", "op": "outer", "m": 80_000, "k": 80_000, "n": 80_000, "rows": "powerlaw",
         "lo": 1, "hi": 8_000},
        # one small factor update, odd dimensions and rank
        {"name": "mttkrp_50k_r20", "op": "mttkrp", "i": 1_201, "j": 907, "k": 701, "nnz": 50_000, "r": 20},
        # the MTTKRP benchmark
        {"name": "mttkrp_20m_r32", "op": "mttkrp", "i": 50_000, "j": 40_000, "k": 30_000, "nnz": 20_000_000, "r": 32},
        # one small tensor-times-matrix, odd dimensions, a rank over 16
        {"name": "ttm_200k_r24", "op": "ttm", "i": 4_001, "j": 3_203, "k": 299, "nnz": 200_000, "r": 24},
        # the TTM benchmark
        {"name": "ttm_10m_r16", "op": "ttm", "i": 100_000, "j": 80_000, "k": 2_000, "nnz": 10_000_000, "r": 16},
        # the transpose pass of the non-fused transposed product
        {"name": "transpose_200k_32", "op": "transpose", "m": 200_000, "n": 200_000, "lo": 32, "hi": 32},
        # a queue of requests served by the batched loop: sizes over the
        # serving mix, half uniform rows and half power-law rows
        {"name": "serve_64", "op": "serve", "count": 64, "lo": 256, "hi": 16_384},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["rowwise", "rowwise", "outer", "mttkrp", "ttm", "transpose", "serve"])
    if op == "rowwise":
        n = _size(rng, 256, 65_536)
        k = max(64, int(n * rng.uniform(0.7, 1.0)))
        m = max(64, int(n * rng.uniform(0.7, 1.0)))
        if rng.random() < 0.5:
            lo = rng.randint(1, 16)
            return {"op": op, "m": m, "k": k, "n": n, "rows": "uniform", "lo": lo, "hi": rng.randint(lo, 48)}
        return {"op": op, "m": m, "k": k, "n": n, "rows": "powerlaw", "lo": 1, "hi": min(4096, n // 4)}
    if op == "outer":
        if rng.random() < 0.5:
            k = _size(rng, 1_000, 30_000)
            return {"op": op, "m": int(k * rng.uniform(0.5, 2.0)), "k": k, "n": int(k * rng.uniform(0.5, 2.0)),
                    "rows": "uniform", "lo": 2, "hi": rng.randint(2, 32)}
        n = _size(rng, 2_000, 60_000)
        return {"op": op, "m": n, "k": n, "n": n, "rows": "powerlaw", "lo": 1, "hi": n // 10}
    if op in ("mttkrp", "ttm"):
        big = op == "mttkrp"
        nnz = _size(rng, 20_000, 20_000_000 if big else 10_000_000)
        f = math.sqrt(nnz / (20e6 if big else 10e6))
        dims = (50_000, 40_000, 30_000) if big else (100_000, 80_000, 2_000)
        i, j, k = (max(200, int(d * f * rng.uniform(0.7, 1.0))) for d in dims)
        return {"op": op, "i": i, "j": j, "k": k, "nnz": nnz, "r": rng.choice([8, 11, 16, 24, 32] if nnz > 5_000_000
                                                                              else [8, 11, 16, 24, 32, 50, 64])}
    if op == "transpose":
        m = _size(rng, 1_000, 200_000)
        lo = rng.randint(1, 16)
        return {"op": op, "m": m, "n": _size(rng, 1_000, 200_000), "lo": lo, "hi": rng.randint(lo, 32)}
    return {"op": op, "count": rng.randint(8, 64), "lo": 256, "hi": _size(rng, 2_048, 16_384)}


# ------------------------------------------------------------------ inputs

_KEPT = {}


def _ctx():
    """The program's context, and the engines its request loop runs on."""
    if "ctx" not in _KEPT:
        _KEPT["ctx"] = Context(0)
    return _KEPT["ctx"]


def _engines():
    if "engines" not in _KEPT:
        ctx = Context(0)
        shape = autotune.apply(ctx, autotune.load())
        caps = serve.default_caps(max_requests=128, max_rows=1 << 20, max_nnz=1 << 25, max_products=1 << 28)
        _KEPT["engines"] = (ctx, [serve.Engine(ctx, caps) for _ in range(shape["engines"])], shape)
    return _KEPT["engines"]


def _rng(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 64 + stream)
    return g


def _perm(g, n):
    return torch.randperm(n, generator=g, device=DEV)


def _uniform(g, shape, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo


def _zipf_cdf(s, lo, hi):
    cdf = torch.cumsum(torch.arange(lo, hi + 1, device=DEV, dtype=torch.float64) ** -s, 0)
    return cdf / cdf[-1]


def _lengths(g, count, rows, lo, hi):
    """Row lengths: uniform in [lo, hi], or Zipf(1.8) on [lo, hi] (its
    quantiles in random order, so that the work does not hang on the seed)."""
    if rows == "uniform":
        return torch.randint(lo, hi + 1, (count,), generator=g, device=DEV)
    u = (torch.arange(count, device=DEV, dtype=torch.float64) + 0.5) / count
    q = (torch.searchsorted(_zipf_cdf(1.8, lo, hi), u) + lo).clamp(lo, hi)
    return q[_perm(g, count)]


# A case has one pattern; the seed permutes its rows, columns and inner index
# (a tensor's modes) and draws the values, so that every seed's inputs are
# others while the sizes of the results stay what they are.

def _csr(pattern, g, m, n, lengths, prow, pcol):
    """(pos, crd, vals) with uniform columns (each once), values in [-1, 1]."""
    rows = torch.repeat_interleave(torch.arange(m, device=DEV), lengths)
    cols = torch.randint(0, n, (rows.numel(),), generator=pattern, device=DEV)
    key = torch.unique(rows * n + cols)
    key = torch.sort(prow[key // n] * n + pcol[key % n])[0]
    pos = torch.zeros(m + 1, dtype=torch.int32, device=DEV)
    pos[1:] = torch.cumsum(torch.bincount(key // n, minlength=m), 0)
    return pos, (key % n).to(torch.int32), _uniform(g, key.numel())


def _coo3(pattern, g, dims, exps, nnz, lo, hi):
    """nnz distinct coordinates; mode d Zipf(exps[d]) over a random
    permutation of its range, or uniform (None)."""
    cdfs = [None if s is None else _zipf_cdf(s, 1, d) for d, s in zip(dims, exps)]
    have = torch.empty(0, dtype=torch.int64, device=DEV)
    for _ in range(60):
        part = min(max(4 * nnz, 1 << 16), 1 << 26)
        key = torch.zeros(part, dtype=torch.int64, device=DEV)
        for d, cdf in zip(dims, cdfs):
            if cdf is None:
                at = torch.randint(0, d, (part,), generator=pattern, device=DEV)
            else:
                u = torch.rand(part, generator=pattern, device=DEV, dtype=torch.float64)
                at = torch.searchsorted(cdf, u).clamp_(max=d - 1)
            key = key * d + at
        have = torch.unique(torch.cat([have, torch.unique(key)]))
        if have.numel() >= nnz:
            break
    if have.numel() > nnz:
        have = have[_perm(pattern, have.numel())[:nnz]]
    idx = (have // (dims[1] * dims[2]), have // dims[2] % dims[1], have % dims[2])
    return [_perm(g, d)[at] for d, at in zip(dims, idx)], _uniform(g, have.numel(), lo, hi)


def _csf(a, b, c, vals, nb, nc):
    """The CSF of a COO with levels a, b, c (torch tensors)."""
    key = (a * nb + b) * nc + c
    key, perm = torch.sort(key)
    ab, fcount = torch.unique_consecutive(key // nc, return_counts=True)
    roots, rcount = torch.unique_consecutive(ab // nb, return_counts=True)

    def starts(count):
        p = torch.zeros(count.numel() + 1, dtype=torch.int32, device=DEV)
        p[1:] = torch.cumsum(count, 0)
        return p

    i32 = torch.int32
    return (roots.to(i32), starts(rcount), (ab % nb).to(i32), starts(fcount), (key % nc).to(i32), vals[perm])


def _tensor(case, seed):
    """COO and factors of a tensor case."""
    g = _rng(seed, 3)
    dims = (case["i"], case["j"], case["k"])
    if case["op"] == "mttkrp":
        idx, vals = _coo3(_rng(0, 4), g, dims, (1.5, 1.5, 1.5), case["nnz"], 0.0, 1.0)
        return idx, vals, _uniform(g, (dims[1], case["r"]), 0.0, 1.0), _uniform(g, (dims[2], case["r"]), 0.0, 1.0)
    idx, vals = _coo3(_rng(0, 4), g, dims, (1.5, 1.5, None), case["nnz"], -1.0, 1.0)
    return idx, vals, None, _uniform(g, (dims[2], case["r"]))


def _operands(case, seed):
    """The two matrices of a product: A's rows (outer: A's columns) and B's."""
    pattern, g = _rng(0, 1), _rng(seed, 1)
    m, k, n = case["m"], case["k"], case["n"]
    lengths = lambda count: _lengths(pattern, count, case["rows"], case["lo"], case["hi"])
    pm, pk, pn = _perm(g, m), _perm(g, k), _perm(g, n)
    b = _csr(pattern, g, k, n, lengths(k), pk, pn)
    if case["op"] == "rowwise":
        return _csr(pattern, g, m, k, lengths(m), pm, pk), b
    if case["rows"] == "powerlaw":
        return b, b  # A = B^T
    return _csr(pattern, g, k, m, lengths(k), pk, pm), b


def _requests(case, seed):
    """The requests' operands: sizes spread evenly over the logarithm of the
    range in random order, uniform 2..64 and power-law rows in turn."""
    pattern, g = _rng(0, 5), _rng(seed, 5)
    count, lo, hi = case["count"], case["lo"], case["hi"]
    out = []
    for t in _perm(pattern, count).tolist():
        n = int(lo * (hi / lo) ** ((t + 0.5) / count))
        rows = ("uniform", 2, min(64, n)) if t % 2 == 0 else ("powerlaw", 1, min(4096, n))
        pm, pk, pn = _perm(g, n), _perm(g, n), _perm(g, n)
        a = _csr(pattern, g, n, n, _lengths(pattern, n, *rows), pm, pk)
        out.append((n, a, _csr(pattern, g, n, n, _lengths(pattern, n, *rows), pk, pn)))
    return out


def _matrix(case, seed):
    pattern, g = _rng(0, 2), _rng(seed, 2)
    m, n = case["m"], case["n"]
    return _csr(pattern, g, m, n, _lengths(pattern, m, "uniform", case["lo"], case["hi"]), _perm(g, m), _perm(g, n))


_NP = {torch.int32: np.int32, torch.int64: np.int64, torch.float64: np.float64}


def _dev(ctx, t):
    """A torch tensor's memory as the device array the entry points take."""
    return DeviceArray.view(ctx, t.data_ptr(), t.numel(), _NP[t.dtype])


class _Lent:
    """A device array as an object that torch can view."""

    def __init__(self, a):
        self.__cuda_array_interface__ = {"shape": (a.count,), "typestr": a.dtype.str, "data": (a.ptr, False),
                                         "version": 2}


def _torch(a):
    if a.count == 0:
        return torch.empty(0, dtype={4: torch.int32, 8: torch.float64}[a.dtype.itemsize], device=DEV)
    return torch.as_tensor(_Lent(a), device=DEV)


def prepare(case, seed):
    op = case["op"]
    ctx = _ctx()
    if op == "rowwise":
        a, b = _operands(case, seed)
        return {"op": op, "kept": (a, b), "ctx": ctx,
                "A": DeviceCSR(case["m"], case["k"], a[1].numel(), *(_dev(ctx, t) for t in a)),
                "B": DeviceCSR(case["k"], case["n"], b[1].numel(), *(_dev(ctx, t) for t in b))}
    if op == "outer":
        a, b = _operands(case, seed)
        k = case["k"]
        # a power-law operand comes compressed in both levels (no row is empty)
        l1 = torch.arange(k, dtype=torch.int32, device=DEV) if case["rows"] == "powerlaw" else None
        up = lambda x: DeviceDCSR(k, None if l1 is None else _dev(ctx, l1), *(_dev(ctx, t) for t in x))
        return {"op": op, "kept": (a, b, l1), "ctx": ctx, "A": up(a), "B": up(b), "dims": (case["m"], k, case["n"])}
    if op in ("mttkrp", "ttm"):
        (i, j, k), vals, bf, cf = _tensor(case, seed)
        if op == "mttkrp":
            x = _csf(j, k, i, vals, case["k"], case["i"])
        else:
            x = _csf(i, k, j, vals, case["k"], case["j"])
        X = DeviceCSF(x[0].numel(), x[2].numel(), x[4].numel(), *(_dev(ctx, t) for t in x))
        return {"op": op, "kept": (x, bf, cf), "ctx": ctx, "X": X, "dims": (case["i"], case["j"], case["k"], case["r"]),
                "factors": [_dev(ctx, f.view(-1)) for f in (bf, cf) if f is not None]}
    if op == "transpose":
        a = _matrix(case, seed)
        nnz = a[1].numel()
        out = (torch.empty(case["n"] + 1, dtype=torch.int32, device=DEV),
               torch.empty(nnz, dtype=torch.int32, device=DEV), torch.empty(nnz, dtype=torch.float64, device=DEV))
        return {"op": op, "ctx": ctx, "a": a, "out": out, "dims": (case["m"], case["n"], nnz)}
    ctx, engines, shape = _engines()
    mats = _requests(case, seed)
    bounds = []
    for n, a, b in mats:
        ends = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV),
                          torch.cumsum((b[0][1:] - b[0][:-1])[a[1].long()], 0)])
        per_row = ends[a[0][1:].long()] - ends[a[0][:-1].long()]
        bounds.append((int(ends[-1]), int(per_row.max())))
    # one output pool for the queue: every request's part sized by its bound
    pos = torch.zeros(sum(n + 1 for n, _, _ in mats), dtype=torch.int32, device=DEV)
    crd = torch.zeros(sum(p for p, _ in bounds), dtype=torch.int32, device=DEV)
    val = torch.zeros(crd.numel(), dtype=torch.float64, device=DEV)
    reqs, at_pos, at = [], 0, 0
    for (n, a, b), (total, longest) in zip(mats, bounds):
        A = DeviceCSR(n, n, a[1].numel(), *(_dev(ctx, t) for t in a))
        B = DeviceCSR(n, n, b[1].numel(), *(_dev(ctx, t) for t in b))
        reqs.append(serve.DeviceRequest(n, n, n, A, B, total, longest, _dev(ctx, pos[at_pos:at_pos + n + 1]),
                                        _dev(ctx, crd[at:at + total]), _dev(ctx, val[at:at + total]), total))
        at_pos += n + 1
        at += total
    return {"op": op, "ctx": ctx, "kept": mats, "reqs": reqs, "out": (pos, crd, val), "engines": engines,
            "arrivals": np.zeros(len(reqs)),
            "shape": {s: shape[s] for s in ("max_batch_products", "large_products", "large_engines")}}


def run(s):
    op, ctx = s["op"], s["ctx"]
    if op == "rowwise":
        c = spgemm_rowwise(ctx, s["A"], s["B"])
        return _torch(c.pos), _torch(c.crd), _torch(c.vals)
    if op == "outer":
        c = spgemm_outer(ctx, s["A"], s["B"], *s["dims"])
        return _torch(c.pos), _torch(c.crd), _torch(c.vals)
    if op == "mttkrp":
        rows, m = mttkrp(ctx, s["X"], *s["dims"], *s["factors"])
        return _torch(rows), _torch(m)
    if op == "ttm":
        fi, fj, y = ttm(ctx, s["X"], *s["dims"], *s["factors"])
        return _torch(fi), _torch(fj), _torch(y)
    if op == "transpose":
        check(lib().spws_csr_transpose_dev(ctx.h, *s["dims"], *(t.data_ptr() for t in s["a"]),
                                           *(t.data_ptr() for t in s["out"])))
        return s["out"]
    _, _, _, nnz = serve.serve(ctx, s["engines"], s["reqs"], s["arrivals"], "batched", with_nnz=True, **s["shape"])
    return (nnz, *s["out"])


# ------------------------------------------------------------- work, exact

def _np_lengths(count, rows, lo, hi):
    if rows == "uniform":
        return np.full(count, (lo + hi) / 2.0)
    cdf = np.cumsum(np.arange(lo, hi + 1, dtype=np.float64) ** -1.8)
    return np.searchsorted(cdf / cdf[-1], (np.arange(count) + 0.5) / count) + float(lo)


def _product_work(m, k, n, rows, lo, hi, outer=False):
    """Expected (nnz(A), nnz(B), products, nnz(C)) of a product."""
    lb = _np_lengths(k, rows, lo, hi)
    if outer:
        # entry (j, i) of A brings B's row j: products = sum_j len_A(j) len_B(j)
        la = lb
        products = float((la * lb).sum())
        # rows of C: each holds about products / m of n columns
        nc = m * n * -math.expm1(-products / (float(m) * n))
    else:
        la = _np_lengths(m, rows, lo, hi)
        products = float(la.sum() * lb.mean())
        nc = float((n * -np.expm1(-la * lb.mean() / n)).sum())
    return float(la.sum()), float(lb.sum()), products, nc


def _tensor_fibers(case):
    """Expected distinct (level 1, level 2) pairs and, for TTM, (i, j) pairs
    of nnz distinct Zipf coordinates, over 48 bins of ranks per mode."""
    def bins(d, s):
        e = np.unique(np.round(np.geomspace(1, d + 1, 48)).astype(np.int64))
        p = np.arange(1, d + 1, dtype=np.float64) ** -s
        c = np.concatenate([[0.0], np.cumsum(p / p.sum())])
        n = np.diff(e).astype(np.float64)
        return n, np.diff(c[e - 1]) / n
    mt = case["op"] == "mttkrp"
    i, j, k = bins(case["i"], 1.5), bins(case["j"], 1.5), bins(case["k"], 1.5 if mt else 0.0)
    n3 = i[0][:, None, None] * j[0][None, :, None] * k[0][None, None, :]
    p3 = i[1][:, None, None] * j[1][None, :, None] * k[1][None, None, :]
    lo, hi = float(case["nnz"]), 1e15
    for _ in range(60):
        mid = math.sqrt(lo * hi)
        lo, hi = (mid, hi) if (n3 * -np.expm1(-mid * p3)).sum() < case["nnz"] else (lo, mid)
    pairs = lambda a, b: float((np.outer(a[0], b[0]) * -np.expm1(-lo * np.outer(a[1], b[1]))).sum())
    return pairs(j, k) if mt else pairs(i, k), pairs(i, j)


def work(case):
    op = case["op"]
    if op in ("rowwise", "outer"):
        na, nb, products, nc = _product_work(case["m"], case["k"], case["n"], case["rows"], case["lo"], case["hi"],
                                             op == "outer")
        rows = 4 * (case["m"] + case["k"]) + (8 if op == "outer" else 4) * case["m"]
        return {"bytes": int(rows + 12 * (na + nb + nc)), "flops": int(2 * products)}
    if op in ("mttkrp", "ttm"):
        fibers, ij = _tensor_fibers(case)
        nnz, r = case["nnz"], case["r"]
        if op == "mttkrp":
            return {"bytes": int(12 * nnz + 8 * fibers + 8 * r * (case["i"] + case["j"] + case["k"])),
                    "flops": int(3 * nnz * r)}
        return {"bytes": int(12 * nnz + 8 * fibers + 8 * r * case["k"] + (8 + 8 * r) * ij), "flops": int(2 * nnz * r)}
    if op == "transpose":
        nnz = case["m"] * (case["lo"] + case["hi"]) / 2.0
        return {"bytes": int(24 * nnz + 4 * (case["m"] + case["n"])), "flops": 0}
    total = {"bytes": 0, "flops": 0}
    for t in range(case["count"]):
        n = int(case["lo"] * (case["hi"] / case["lo"]) ** ((t + 0.5) / case["count"]))
        rows = ("uniform", 2, min(64, n)) if t % 2 == 0 else ("powerlaw", 1, min(4096, n))
        na, nb, products, nc = _product_work(n, n, n, *rows)
        total["bytes"] += int(12 * n + 12 * (na + nb + nc))
        total["flops"] += int(2 * products)
    return total


def _exact_product(a, b, m, n):
    """Sorted CSR of A * B in plain torch: rows in blocks, each block's
    products added into a dense array."""
    ap, ai, ax = a
    bp, bi, bx = b
    ap, bp = ap.long(), bp.long()
    lens = (bp[1:] - bp[:-1])[ai.long()]
    ends = torch.zeros(ai.numel() + 1, dtype=torch.int64, device=DEV)
    ends[1:] = torch.cumsum(lens, 0)
    row_of = torch.repeat_interleave(torch.arange(m, device=DEV), ap[1:] - ap[:-1])
    at_row = ends[ap].cpu().numpy()   # products before each row
    ap_host = ap.cpu().numpy()
    counts, crd, vals = [], [], []
    r0 = 0
    while r0 < m:
        r1 = max(r0 + 1, min(m, r0 + (1 << 28) // max(n, 1)))
        r1 = max(r0 + 1, min(r1, int(np.searchsorted(at_row, at_row[r0] + (1 << 28), side="right")) - 1))
        e0, e1 = int(ap_host[r0]), int(ap_host[r1])
        acc = torch.zeros((r1 - r0) * n, dtype=torch.float64, device=DEV)
        seen = torch.zeros((r1 - r0) * n, dtype=torch.bool, device=DEV)
        if e1 > e0:
            own = torch.repeat_interleave(torch.arange(e0, e1, device=DEV), lens[e0:e1])
            src = torch.arange(own.numel(), device=DEV) - (ends[own] - ends[e0]) + bp[ai[own].long()]
            at = (row_of[own] - r0) * n + bi[src].long()
            acc.index_add_(0, at, ax[own] * bx[src])
            seen[at] = True
        hit = torch.nonzero(seen).view(-1)
        counts.append(torch.bincount(hit // n, minlength=r1 - r0))
        crd.append((hit % n).to(torch.int32))
        vals.append(acc[hit])
        r0 = r1
    pos = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    pos[1:] = torch.cumsum(torch.cat(counts), 0)
    return pos, torch.cat(crd), torch.cat(vals)


def _transposed(a, m, n):
    """The n x m transpose of an m x n CSR, in plain torch."""
    rows = torch.repeat_interleave(torch.arange(m, device=DEV), (a[0][1:] - a[0][:-1]).long())
    key, perm = torch.sort(a[1].long() * m + rows)
    pos = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    pos[1:] = torch.cumsum(torch.bincount(key // m, minlength=n), 0)
    return pos, (key % m).to(torch.int32), a[2][perm]


def exact(case, seed):
    op = case["op"]
    if op == "rowwise":
        a, b = _operands(case, seed)
        pos, crd, vals = _exact_product(a, b, case["m"], case["n"])
        return pos.to(torch.int32), crd, vals
    if op == "outer":
        a, b = _operands(case, seed)
        return _exact_product(_transposed(a, case["k"], case["m"]), b, case["m"], case["n"])
    if op == "transpose":
        a = _matrix(case, seed)
        return _transposed(a, case["m"], case["n"])
    if op in ("mttkrp", "ttm"):
        (i, j, k), vals, bf, cf = _tensor(case, seed)
        if op == "mttkrp":
            rows, to, count = torch.unique(i), i, case["i"]
        else:
            rows, to = torch.unique(i * case["j"] + j, return_inverse=True)
            count = rows.numel()
        out = torch.zeros((count, case["r"]), dtype=torch.float64, device=DEV)
        for at in range(0, vals.numel(), 1 << 22):
            p = slice(at, at + (1 << 22))
            part = vals[p, None] * cf[k[p]]
            out.index_add_(0, to[p], part if bf is None else part * bf[j[p]])
        if op == "mttkrp":
            return rows.to(torch.int32), out.view(-1)
        return (rows // case["j"]).to(torch.int32), (rows % case["j"]).to(torch.int32), out.view(-1)
    mats = _requests(case, seed)
    nnz, pos, crd, val = [], [], [], []
    for n, a, b in mats:
        p, c, v = _exact_product(a, b, n, n)
        room = int((b[0][1:] - b[0][:-1])[a[1].long()].sum()) - c.numel()
        nnz.append(c.numel())
        pos.append(p.to(torch.int32))
        crd += [c, torch.zeros(room, dtype=torch.int32, device=DEV)]
        val += [v, torch.zeros(room, dtype=torch.float64, device=DEV)]
    return np.array(nnz, dtype=np.int64), torch.cat(pos), torch.cat(crd), torch.cat(val)
