"""The work that programs have this framework do, as measurable cases.

A case is a dict of plain values. ``listed()`` names the fixed ones, ``draw``
makes more of the same ranges, ``prepare`` builds what a program holds before
its call (graphs resident in device memory, weights, request lists, servers,
captured batches), ``run`` makes one pass through the public entry points,
``work`` is what a pass cannot do without, and ``exact`` is the same result in
64-bit arithmetic from plain torch operations.

Graph families and sizes are those of bench.py, the batched and served
workloads (jaccard_amd/batch.py, jaccard_amd/serve.py) and the tests: RMAT
(.57/.19/.19) from 2^8 to 2^22 vertices with edge factors 4 to 32, and the
Chung-Lu power law (exponent 2.1, mean degree 32). Graphs are symmetric, free
of self loops and duplicates, rows sorted, weights float32 uniform in (0, 1],
the same in both directions of an edge.
"""
from __future__ import annotations

import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sycl-jaccard_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from jaccard_amd import api, batch, graphs, serve  # noqa: E402

DEV = "cuda"


# ---- cases -------------------------------------------------------------------

def _graph(name, family, n, ef, weighted, algo="ec", symmetric=False):
    return {"name": name, "kind": "graph", "family": family, "n": n, "ef": ef, "weighted": weighted, "algo": algo,
            "symmetric": symmetric}


def listed():
    return [
        # one graph of the low end of the 4096-graph set, called alone: a
        # program with small graphs pays mostly launches
        _graph("ec_n700", "rmat", 700, 8, False),
        # a mid-sized member of that set, weighted as half of them are (vertex
        # weights from edge weights, then the weighted coefficients)
        _graph("weighted_n9001", "rmat", 9001, 17, True),
        # the plain edge-centric configuration (RMAT-16, unweighted)
        _graph("ec_rmat16", "rmat", 1 << 16, 16, False),
        # the vertex-centric pipeline of a graph its program knows to be
        # symmetric, at an odd size
        _graph("vc_weighted_n200003", "rmat", 200003, 16, True, algo="vc", symmetric=True),
        # the skewed power-law graph
        _graph("ec_chunglu20", "chunglu", 1 << 20, 32, False),
        # the headline: RMAT-22, weighted, edge-centric, as the driver calls it
        _graph("weighted_rmat22", "rmat", 1 << 22, 16, True),
        # a program written against the kernel-level entry points (row sum,
        # fill, intersection, weight), fp32 buffers
        {"name": "kernels_n150001", "kind": "kernels", "n": 150001, "ef": 16},
        # queries of a handful of vertex pairs against a resident graph, as a
        # link-prediction loop makes them one after another
        {"name": "pairs_64", "kind": "pairs", "n": 1 << 15, "ef": 16, "pairs": 64, "weighted": False},
        # the largest pair query of the serving mix, alone
        {"name": "pairs_weighted_65536", "kind": "pairs", "n": 1 << 18, "ef": 16, "pairs": 65536, "weighted": True},
        # many small graphs in one captured launch (a slice of the 4096-graph
        # workload, half of them weighted)
        {"name": "batch_128", "kind": "batch", "count": 128},
        # a burst of whole-graph and pair requests against resident graphs
        {"name": "serve_burst_96", "kind": "serve", "graphs": 10, "smin": 12, "smax": 16, "requests": 96},
        # building the graph on the device from raw draws, with edge weights
        {"name": "ingest_n1000003", "kind": "ingest", "n": 1000003, "ef": 16, "weighted": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["graph", "graph", "graph", "graph", "kernels", "pairs", "batch", "serve", "ingest"])
    if kind == "graph":
        if rng.random() < 0.25:
            n = _log_int(rng, 1 << 14, 1 << 20) | 1
            c = _graph("", "chunglu", n, rng.randint(8, 32), rng.random() < 0.5)
        else:
            n = _log_int(rng, 300, 1 << 21)
            c = _graph("", "rmat", n, rng.randint(4, 32 if n < (1 << 18) else 16), rng.random() < 0.5)
        c["algo"] = "vc" if rng.random() < 0.25 else "ec"
        c["symmetric"] = rng.random() < 0.4
    elif kind == "kernels":
        c = {"kind": kind, "n": _log_int(rng, 1000, 1 << 19), "ef": rng.randint(4, 24)}
    elif kind == "pairs":
        c = {"kind": kind, "n": _log_int(rng, 1 << 14, 1 << 20), "ef": 16, "pairs": _log_int(rng, 1, 65536),
             "weighted": rng.random() < 0.5}
    elif kind == "batch":
        c = {"kind": kind, "count": _log_int(rng, 8, 160)}
    elif kind == "serve":
        smin = rng.randint(12, 14)
        c = {"kind": kind, "graphs": rng.randint(4, 12), "smin": smin, "smax": smin + rng.randint(1, 3),
             "requests": _log_int(rng, 16, 128)}
    else:
        c = {"kind": kind, "n": _log_int(rng, 1000, 1 << 21), "ef": rng.randint(4, 16), "weighted": rng.random() < 0.5}
    c.pop("name", None)
    return c


# ---- inputs ------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _pairs_of(n, ef):
    """Undirected edges of an RMAT graph of n vertices and ef * n draws (about
    what merging repeats leaves), the same for every seed."""
    return int(ef * n * max(0.4, 1.0 - 2.1 * math.sqrt(ef / 16.0) * n ** -0.25))


def _rmat_draws(n, e, gen):
    """About e RMAT draws below n (int64 source and target)."""
    scale = max(1, math.ceil(math.log2(n)))
    if n != 1 << scale:
        e = int(1.6 * e)
    s = torch.zeros(e, dtype=torch.int32, device=DEV)
    d = torch.zeros(e, dtype=torch.int32, device=DEV)
    for _ in range(scale):
        r = torch.rand(e, generator=gen, device=DEV)
        row = r >= graphs.RMAT_A + graphs.RMAT_B
        col = ((r >= graphs.RMAT_A) & ~row) | (r >= graphs.RMAT_A + graphs.RMAT_B + graphs.RMAT_C)
        s = s * 2 + row
        d = d * 2 + col
    ok = (s < n) & (d < n) & (s != d)
    return s[ok].long(), d[ok].long()


def _chunglu_cdf(n, mean):
    """Running sum of power-law endpoint weights (exponent 2.1, largest
    expected degree 2^17 or n / 8)."""
    beta = 1.0 / 1.1
    top = float(min(1 << 17, n // 8))
    i = torch.arange(n, dtype=torch.float64, device=DEV)
    lo, hi = 1e-6, 1e9
    for _ in range(48):
        mid = math.sqrt(lo * hi)
        if float((top * (1.0 + i / mid) ** -beta).mean()) < mean:
            lo = mid
        else:
            hi = mid
    return torch.cumsum((1.0 + i / math.sqrt(lo * hi)) ** -beta, 0)


def _edges(family, n, ef, gen):
    """The graph's undirected edges, as sorted keys low * n + high."""
    want = _pairs_of(n, ef) if family == "rmat" else n * ef // 2
    cdf = _chunglu_cdf(n, ef) if family == "chunglu" else None
    keys, more = None, int(1.1 * (ef * n if family == "rmat" else want)) + 64
    while keys is None or keys.numel() < want:
        if family == "rmat":
            s, d = _rmat_draws(n, more, gen)
        else:
            s, d = (torch.searchsorted(cdf, torch.rand(more, generator=gen, device=DEV, dtype=torch.float64) * cdf[-1])
                    .clamp_(max=n - 1) for _ in range(2))
            s, d = s[s != d], d[s != d]
        k = torch.minimum(s, d) * n + torch.maximum(s, d)
        keys = torch.unique(k if keys is None else torch.cat([keys, k]))
        more = int(0.2 * more) + 64
    if keys.numel() > want:
        keys = torch.sort(keys[torch.randperm(keys.numel(), generator=gen, device=DEV)[:want]]).values
    return keys


def _csr(n, und, gen, weighted):
    """Symmetric sorted CSR (offsets, indices, weights or None) of undirected
    keys low * n + high."""
    a, b = und // n, und % n
    keys, order = torch.sort(torch.cat([und, b * n + a]))
    rows = keys // n
    ind = (keys - rows * n).to(torch.int32)
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    w = None
    if weighted:
        uw = 1.0 - torch.rand(und.numel(), generator=gen, device=DEV)
        w = torch.cat([uw, uw])[order].contiguous()
    return off.to(torch.int32), ind.contiguous(), w


def _device_graph(case, seed, weighted):
    gen = _gen(seed)
    und = _edges(case.get("family", "rmat"), case["n"], case["ef"], gen)
    return api.DeviceCSR(case["n"], *_csr(case["n"], und, gen, weighted)), gen


def _vertex_weights64(off, ind, w):
    """fp64 sum of each row's edge weights."""
    n = off.numel() - 1
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), (off[1:] - off[:-1]).long())
    return torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, rows, w.double())


def _pair_draws(off, ind, k, gen):
    """Half stored edges, half uniform random pairs of vertices with an edge."""
    n, deg = off.numel() - 1, (off[1:] - off[:-1]).long()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV, dtype=torch.int32), deg)
    e = torch.randint(0, ind.numel(), (k // 2,), generator=gen, device=DEV)
    live = torch.nonzero(deg).flatten().to(torch.int32)
    r = live[torch.randint(0, live.numel(), (2, k - k // 2), generator=gen, device=DEV)]
    perm = torch.randperm(k, generator=gen, device=DEV)
    return torch.cat([rows[e], r[0]])[perm].contiguous(), torch.cat([ind[e], r[1]])[perm].contiguous()


def _host_graph(n, off, ind, w):
    return graphs.CSRGraph(n, off.cpu().numpy(), ind.cpu().numpy(), None if w is None else w.cpu().numpy())


def _batch_unions(case, seed):
    """(offsets, indices, weights or None, first vertices, first entries) of
    the unweighted and of the weighted half: the members of the batched
    workload's sizes, packed with global ids."""
    gen = _gen(seed)
    ns, efs, _, wts = batch.batch_specs(case["count"], 1)
    out = []
    for weighted in (False, True):
        members = [(int(n), int(ef)) for n, ef, w in zip(ns, efs, wts) if bool(w) == weighted]
        vbase = np.cumsum([0] + [n for n, _ in members])
        ebase = np.cumsum([0] + [2 * _pairs_of(n, ef) for n, ef in members])
        total = int(vbase[-1])
        und = []
        for (n, ef), v0 in zip(members, vbase):
            k = _edges("rmat", n, ef, gen)
            und.append((k // n + int(v0)) * total + k % n + int(v0))
        out.append(_csr(total, torch.cat(und), gen, weighted) + (vbase, ebase))
    return out


def _serve_inputs(case, seed):
    """Resident graphs (scales cycling) and a burst of requests, half of them
    whole-graph, the others k pairs, k log-uniform in [1, 65536]."""
    gen, rng = _gen(seed), random.Random(case["requests"])
    gs = []
    for i in range(case["graphs"]):
        n = 1 << (case["smin"] + i % (case["smax"] - case["smin"] + 1))
        gs.append((n,) + _csr(n, _edges("rmat", n, 16, gen), gen, True))
    reqs = []
    for i in range(case["requests"]):
        gi = rng.randrange(len(gs))
        if i % 2 == 0:
            reqs.append(serve.Request(gi, serve.REQ_FULL, 0.0))
        else:
            f, s = _pair_draws(gs[gi][1], gs[gi][2], _log_int(rng, 1, 65536), gen)
            reqs.append(serve.Request(gi, serve.REQ_PAIRS, 0.0, f.cpu().numpy(), s.cpu().numpy()))
    return gs, reqs


def prepare(case, seed):
    kind = case["kind"]
    if kind == "graph":
        g, _ = _device_graph(case, seed, case["weighted"])
        return {"case": case, "g": g}
    if kind == "kernels":
        g, _ = _device_graph(case, seed, True)
        return {"case": case, "g": g, "v": api.vertex_weights(g)}
    if kind == "pairs":
        g, gen = _device_graph(case, seed, case["weighted"])
        first, second = _pair_draws(g.offsets, g.indices, case["pairs"], gen)
        return {"case": case, "g": g, "first": first, "second": second,
                "W": api.vertex_weights(g) if case["weighted"] else None}
    if kind == "batch":
        parts = [batch.GraphBatch(_host_graph(off.numel() - 1, off, ind, w), vbase, ebase, np.arange(len(vbase) - 1))
                 for off, ind, w, vbase, ebase in _batch_unions(case, seed)]
        runner = batch.BatchRunner(parts, DEV)
        runner.select()
        runner.capture()
        return {"case": case, "runner": runner}
    if kind == "serve":
        gs, reqs = _serve_inputs(case, seed)
        gs = [_host_graph(*g) for g in gs]
        # one result buffer per graph, pair results side by side
        full = {q.graph: torch.empty(gs[q.graph].m, dtype=torch.float32, device=DEV) for q in reqs if not q.num_pairs}
        pairs = torch.empty(sum(q.num_pairs for q in reqs), dtype=torch.float32, device=DEV)
        results, at = [], 0
        for q in reqs:
            results.append(pairs[at:at + q.num_pairs] if q.num_pairs else full[q.graph])
            at += q.num_pairs
        return {"case": case, "server": serve.Server(gs, DEV), "reqs": reqs, "results": results,
                "out": [full[i] for i in sorted(full)] + [pairs]}
    # raw draws: every edge at least once, a part of them again, either way
    # round, in no order, with a few self loops
    gen, n = _gen(seed), case["n"]
    und = _edges("rmat", n, case["ef"], gen)
    again = torch.randint(0, und.numel(), (case["n"] * case["ef"] - und.numel(),), generator=gen, device=DEV)
    k = torch.cat([und, und[again]])
    k = k[torch.randperm(k.numel(), generator=gen, device=DEV)]
    a, b = k // n, k % n
    turn = torch.rand(k.numel(), generator=gen, device=DEV) < 0.5
    src, dst = torch.where(turn, b, a).to(torch.int32), torch.where(turn, a, b).to(torch.int32)
    loops = torch.arange(0, n, 97, dtype=torch.int32, device=DEV)
    src, dst = torch.cat([src, loops]), torch.cat([dst, loops])
    w = 1.0 - torch.rand(src.numel(), generator=gen, device=DEV) if case["weighted"] else None
    return {"case": case, "src": src, "dst": dst, "w": w}


# ---- one pass ----------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "graph":
        g = state["g"]
        flags = api.FLAG_ASSUME_SYMMETRIC if case["symmetric"] else 0
        ec = case["algo"] == "ec"
        if not case["weighted"]:
            return api.jaccard(g, edge_centric=ec, flags=flags)
        W = api.vertex_weights(g)
        return W, api.jaccard(g, weights=W, edge_centric=ec, flags=flags)
    if kind == "kernels":
        g = state["g"]
        work = torch.empty(g.n, dtype=torch.float32, device=DEV)
        wi, ws, wj = (torch.empty(g.m, dtype=torch.float32, device=DEV) for _ in range(3))
        api.rowsum(g, work, v=state["v"])
        api.fill(wi, 0.0)
        api.intersect(g, work, wi, ws, v=state["v"])
        api.jw(wi, ws, wj)
        return work, wi, ws, wj
    if kind == "pairs":
        return api.jaccard_list(state["g"], state["first"], state["second"], weights=state["W"])
    if kind == "batch":
        runner = state["runner"]
        runner.replay()
        return [t for it in runner.items for t in ((it["out"],) if it["W"] is None else (it["W"], it["out"]))]
    if kind == "serve":
        state["server"].run(state["reqs"], state["results"])
        return state["out"]
    g = api.csr_from_edges(case["n"], state["src"], state["dst"], state["w"])
    return (g.offsets, g.indices) if g.edge_w is None else (g.offsets, g.indices, g.edge_w)


# ---- what a pass cannot do without ---------------------------------------------

def _graph_work(n, m, weighted):
    # offsets, columns, result; weighted: edge weights read, vertex weights
    # written and read
    b = 4.0 * (n + 1) + 8.0 * m + (4.0 * m + 8.0 * n if weighted else 0.0)
    return b, 3.0 * m


def work(case):
    kind = case["kind"]
    if kind == "graph":
        m = case["n"] * case["ef"] if case["family"] == "chunglu" else 2 * _pairs_of(case["n"], case["ef"])
        b, f = _graph_work(case["n"], m, case["weighted"])
    elif kind == "kernels":
        m = 2 * _pairs_of(case["n"], case["ef"])
        b, f = 4.0 * (3 * case["n"] + 1) + 16.0 * m, 3.0 * m
    elif kind == "pairs":
        # both rows of every pair (a mean row), the pair, the result
        row = 2.0 * _pairs_of(case["n"], case["ef"]) / case["n"]
        b, f = case["pairs"] * (8.0 * row + 12.0), case["pairs"] * (row + 3.0)
    elif kind == "batch":
        ns, efs, _, weighted = batch.batch_specs(case["count"], 1)
        parts = [_graph_work(int(n), 2 * _pairs_of(int(n), int(ef)), bool(w)) for n, ef, w in zip(ns, efs, weighted)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "serve":
        sizes = [1 << (case["smin"] + i % (case["smax"] - case["smin"] + 1)) for i in range(case["graphs"])]
        full = case["requests"] / 2.0 / len(sizes)
        b = full * sum(4.0 * n + 8.0 * 2 * _pairs_of(n, 16) for n in sizes) + case["requests"] / 2.0 * 6000 * 250.0
        f = full * sum(3.0 * 2 * _pairs_of(n, 16) for n in sizes)
    else:
        e = case["n"] * case["ef"]
        m = 2 * _pairs_of(case["n"], case["ef"])
        b, f = 8.0 * e + 4.0 * m + 4.0 * case["n"] + (4.0 * e + 4.0 * m if case["weighted"] else 0.0), 0.0
    return {"bytes": b, "flops": f}


# ---- the same results in 64 bits -------------------------------------------------

def _intersections(off, ind, W, a, b):
    """Per pair (a, b): the fp64 sum of W (None: the count) over the common
    neighbours, by searching each entry of the shorter row in the longer."""
    n = off.numel() - 1
    off = off.long()
    deg = off[1:] - off[:-1]
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    keys = rows * n + ind.long()
    a, b = a.long(), b.long()
    swap = deg[a] > deg[b]
    s, t = torch.where(swap, b, a), torch.where(swap, a, b)
    out = torch.zeros(a.numel(), dtype=torch.float64, device=DEV)
    if keys.numel() == 0:
        return out
    ends = torch.cumsum(deg[s], 0)
    lo = 0
    while lo < a.numel():
        base = int(ends[lo - 1]) if lo else 0
        hi = max(lo + 1, int(torch.searchsorted(ends, base + (1 << 26))))
        d = deg[s[lo:hi]]
        item = torch.repeat_interleave(torch.arange(hi - lo, device=DEV), d)
        pos = torch.arange(item.numel(), device=DEV) - (torch.cumsum(d, 0) - d)[item] + off[s[lo:hi]][item]
        y = ind[pos].long()
        want = t[lo:hi][item] * n + y
        hit = keys[torch.searchsorted(keys, want).clamp_(max=keys.numel() - 1)] == want
        y, item = y[hit], item[hit]
        add = torch.ones(item.numel(), dtype=torch.float64, device=DEV) if W is None else W[y]
        out[lo:hi].index_add_(0, item, add)
        lo = hi
    return out


def _row_sums(off, ind, W):
    n = off.numel() - 1
    deg = (off[1:] - off[:-1]).long()
    if W is None:
        return deg.double()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    return torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, rows, W[ind.long()])


def _edge_values(off, ind, W):
    """(intersection, row sum of both ends) of every stored edge."""
    n = off.numel() - 1
    deg = (off[1:] - off[:-1]).long()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    cols = ind.long()
    one = rows < cols
    I = torch.zeros(ind.numel(), dtype=torch.float64, device=DEV)
    I[one] = _intersections(off, ind, W, rows[one], cols[one])
    # the mirror of entry (v, u): where (u, v) stands among the sorted keys
    I[~one] = I[torch.searchsorted(rows * n + cols, cols[~one] * n + rows[~one])]
    S = _row_sums(off, ind, W)
    return I, S[rows] + S[cols]


def _probes(off, ind):
    deg = (off[1:] - off[:-1]).long()
    rows = torch.repeat_interleave(deg, deg)
    return float(torch.minimum(rows, deg[ind.long()]).sum()) / 2


def exact(case, seed):
    kind = case["kind"]
    if kind in ("graph", "kernels"):
        g, _ = _device_graph(case, seed, kind == "kernels" or case["weighted"])
        if _probes(g.offsets, g.indices) > 4.5e9:
            return None
        W = None if g.edge_w is None else _vertex_weights64(g.offsets, g.indices, g.edge_w)
        I, S = _edge_values(g.offsets, g.indices, W)
        J = I / (S - I)
        if kind == "kernels":
            return _row_sums(g.offsets, g.indices, W), I, S, J
        return J if W is None else (W, J)
    if kind == "pairs":
        g, gen = _device_graph(case, seed, case["weighted"])
        first, second = _pair_draws(g.offsets, g.indices, case["pairs"], gen)
        W = None if g.edge_w is None else _vertex_weights64(g.offsets, g.indices, g.edge_w)
        I = _intersections(g.offsets, g.indices, W, first, second)
        S = _row_sums(g.offsets, g.indices, W)
        return I / (S[first.long()] + S[second.long()] - I)
    if kind == "batch":
        out = []
        for off, ind, w, _, _ in _batch_unions(case, seed):
            if _probes(off, ind) > 4.5e9:
                return None
            W = None
            if w is not None:
                W = _vertex_weights64(off, ind, w)
                out.append(W)
            I, S = _edge_values(off, ind, W)
            out.append(I / (S - I))
        return out
    if kind == "serve":
        gs, reqs = _serve_inputs(case, seed)
        full, pairs = {}, []
        for q in reqs:
            _, off, ind, w = gs[q.graph]
            W = _vertex_weights64(off, ind, w)
            if q.kind == serve.REQ_FULL:
                if q.graph not in full:
                    I, S = _edge_values(off, ind, W)
                    full[q.graph] = I / (S - I)
            else:
                a, b = (torch.from_numpy(x).to(DEV) for x in (q.first, q.second))
                I = _intersections(off, ind, W, a, b)
                S = _row_sums(off, ind, W)
                pairs.append(I / (S[a.long()] + S[b.long()] - I))
        return [full[i] for i in sorted(full)] + [torch.cat(pairs)]
    return None
