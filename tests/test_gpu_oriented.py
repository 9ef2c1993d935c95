"""Oriented engine (triangles of the degree-ranked graph) against the oracle
and, bit for bit, the owner engine: sizes around its tile and table limits,
and the graphs it must refuse (the owner engine then delivers).

Tolerance: counts are integers and weighted sums exact in both engines, so
their results are equal; against the FP64 oracle the weighted results carry
one fp32 rounding (2^-24), bounded by the repository's 1e-6.
"""
import numpy as np
import pytest

import oracle
from jaccard_amd import api, graphs

import cases

pytestmark = pytest.mark.gpu


def grid_weights(n, seed, zero=False):
    """Multiples of 2^-24 in (0, 1]: fp64 sums are exact."""
    w = ((1 + np.random.default_rng(seed).integers(0, 1 << 24, n)) * 2.0 ** -24).astype(np.float32)
    return np.zeros_like(w) if zero else w


def circulant(n, reach):
    """Every vertex next to the `reach` ids on both sides: a regular graph, so
    ranks past 65535 with long rows (the 32-bit wedge kernel)."""
    i = np.repeat(np.arange(n), reach)
    return graphs.from_edges(n, i, (i + np.tile(np.arange(1, reach + 1), n)) % n)


def layers(k, width, seed=5):
    """A clique of k vertices, each also tied to `width` others of its own and
    to random ids: R(u) of up to k - 1 entries, rows of every length class."""
    rng = np.random.default_rng(seed)
    a, b = np.triu_indices(k, 1)
    own = np.repeat(np.arange(k), width)
    tail = k + np.arange(k * width)
    s = rng.integers(0, k, 4 * k)
    return graphs.from_edges(k + k * width, np.concatenate([a, own, s]),
                             np.concatenate([b, tail, k + rng.integers(0, k * width, 4 * k)]))


def asymmetric():
    g = graphs.rmat(11, 16, seed=3)
    rng = np.random.default_rng(4)
    keep = np.sort(rng.choice(g.m, g.m - 40, replace=False))
    rows = np.repeat(np.arange(g.n), np.diff(g.offsets))
    return graphs.from_edges(g.n, rows[keep], g.indices[keep], symmetrize=False)


def self_loop():
    g = graphs.rmat(9, 8, seed=3)
    u = int(np.argmax(np.diff(g.offsets)))
    at = int(g.offsets[u] + np.searchsorted(g.indices[g.offsets[u]:g.offsets[u + 1]], u))
    ind = np.insert(g.indices, at, u).astype(np.int32)
    off = g.offsets.copy()
    off[u + 1:] += 1
    return graphs.CSRGraph(g.n, off, ind)


# name: (graph, engine delivers)
GRAPHS = {
    "k2": (lambda: cases.complete(2), True),
    "k17": (lambda: cases.complete(17), True),
    "k33": (lambda: cases.complete(33), True),
    "k65": (lambda: cases.complete(65), True),
    "k130": (lambda: cases.complete(130), True),
    "star": (lambda: cases.star(1500), True),
    "path": (lambda: cases.path(70), True),
    "bipartite": (lambda: cases.complete_bipartite(20, 1100), True),
    "rmat13_odd": (lambda: graphs.rmat_n(5001, 13.0, 3), True),
    "rmat16": (lambda: graphs.rmat(16, 16, seed=2), True),
    "chunglu": (lambda: graphs.chung_lu(1 << 14, max_deg=4096.0, seed=2), True),
    "layers": (lambda: layers(600, 3), True),
    "rank32": (lambda: circulant(66001, 96), True),
    "k700_matrix_budget": (lambda: cases.complete(700), True),
    "k2000_over_budget": (lambda: cases.complete(2000), False),
    "asymmetric": (asymmetric, False),
    "self_loop": (self_loop, False),
}


def union(weighted):
    """Small graphs side by side, ids without neighbours before, between and
    after them, a part of two vertices, one of 9001."""
    from jaccard_amd import batch
    b = batch.rmat_batch([256, 2, 700, 9001, 300, 4096], [4.0, 1.0, 9.0, 12.0, 30.0, 16.0], [1, 2, 3, 4, 5, 6], weighted)
    g = b.union
    pad = 37
    off = np.concatenate([np.zeros(pad, np.int32), g.offsets, np.full(5, g.offsets[-1], np.int32)])
    return graphs.CSRGraph(g.n + pad + 5, off.astype(np.int32), (g.indices + pad).astype(np.int32))


def run(dg, W, engine, device, members=0):
    """Result and, for the oriented engine, whether it delivered."""
    import torch
    n, m, weighted = dg.n, dg.m, W is not None
    need = api.workspace_size(n, min(m, 1 << 20), weighted, True) if m <= 1 << 20 else 0
    if engine == api.ENGINE_ORIENTED and need:
        ws = torch.zeros(need + 64 * m + 256 * n + (1 << 20), dtype=torch.uint8, device=device)
        out = api.jaccard(dg, weights=W, workspace=ws, tuning=dict(engine=engine, members=members))
        done = int(ws[need + 4:need + 8].view(torch.int32))  # the engine's flag, second word of its area
        return out, done == 1
    return api.jaccard(dg, weights=W, tuning=dict(engine=engine, members=members)), None


def same(a, b):
    import torch
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("name", list(GRAPHS))
def test_oriented_equals_owner_and_oracle(name, cuda):
    make, delivers = GRAPHS[name]
    g = make()
    print(f"[gpu] oriented {name} n={g.n} m={g.m}", flush=True)
    dg = api.DeviceCSR.from_host(g, cuda)
    import torch
    for kind in ("unweighted", "weighted", "zero"):
        W = None if kind == "unweighted" else torch.from_numpy(grid_weights(g.n, 7, kind == "zero")).to(cuda)
        out, done = run(dg, W, api.ENGINE_ORIENTED, cuda)
        own, _ = run(dg, W, api.ENGINE_OWNER, cuda)
        assert same(out, own), kind
        if done is not None:
            assert done == delivers, kind
        host = out.cpu().numpy()
        if g.m > 1 << 21:
            continue  # the owner engine's own tests hold it to the oracle
        if kind == "unweighted":
            assert np.array_equal(host.view(np.uint32), oracle.ec_unweighted(g).view(np.uint32))
        elif kind == "weighted":
            ref = oracle.weighted_f64(g, W.cpu().numpy().astype(np.float64))
            assert np.all(np.abs(host - ref) <= 1e-6 * np.abs(ref))


# name: (graph, engine delivers with every part ranked by itself)
MEMBERS = {
    "union": (lambda: union(False), True),
    "one_graph": (lambda: graphs.rmat(14, 16, seed=4), True),
    "edgeless_tail": (lambda: graphs.from_edges(5000, [0, 1], [1, 2]), True),
    "too_large_a_part": (lambda: cases.star(70000), False),
    "asymmetric": (asymmetric, False),
}


@pytest.mark.parametrize("name", list(MEMBERS))
def test_members(name, cuda):
    make, delivers = MEMBERS[name]
    g = make()
    print(f"[gpu] oriented members {name} n={g.n} m={g.m}", flush=True)
    dg = api.DeviceCSR.from_host(g, cuda)
    import torch
    for W in (None, torch.from_numpy(grid_weights(g.n, 7)).to(cuda)):
        out, done = run(dg, W, api.ENGINE_ORIENTED, cuda, members=1)
        assert done == delivers
        assert same(out, run(dg, W, api.ENGINE_OWNER, cuda)[0])
        if W is None:
            assert np.array_equal(out.cpu().numpy().view(np.uint32), oracle.ec_unweighted(g).view(np.uint32))


def test_kernel_level_intersection(cuda):
    """jc_intersect from its size on: adds into weight_i, writes weight_s, the
    same bits as below that size by the owner engine (a tuning the kernel-level
    entry does not take, so a part of the graph is compared with the oracle)."""
    import torch
    g = graphs.rmat(18, 16, seed=12)
    dg = api.DeviceCSR.from_host(g, cuda)
    for weighted in (False, True):
        v = torch.from_numpy(grid_weights(g.n, 2)).to(cuda) if weighted else None
        work = torch.empty(g.n, dtype=torch.float32, device=cuda)
        wi = torch.full((g.m,), 2.0, dtype=torch.float32, device=cuda)
        ws = torch.empty(g.m, dtype=torch.float32, device=cuda)
        api.rowsum(dg, work, v=v)
        api.intersect(dg, work, wi, ws, v=v)
        rows = np.repeat(np.arange(g.n), np.diff(g.offsets))
        wk = work.cpu().numpy()
        assert np.array_equal(ws.cpu().numpy(), wk[rows] + wk[g.indices])
        # J = I / (S - I) gives I back: the oracle's quotients of the same edges
        e = np.random.default_rng(1).choice(g.m, 20000, replace=False)
        got = wi.cpu().numpy()[e].astype(np.float64) - 2.0
        s = (wk[rows[e]].astype(np.float64) + wk[g.indices[e]])
        if weighted:
            J = oracle.pairs_weighted_f64(g, v.cpu().numpy().astype(np.float64), rows[e], g.indices[e])
        else:
            J = oracle.pairs_unweighted(g, rows[e], g.indices[e]).astype(np.float64)
        I = J / (1.0 + J) * s
        # fp32 row sums, quotient and 2 + I: a few roundings of 2^-24 of I + 2 and S J
        assert np.all(np.abs(got - I) <= 8 * 2.0 ** -24 * (np.abs(I) + 2.0 + s * np.abs(J)))


@pytest.mark.parametrize("name", ["wide", "negative", "infinite", "nan"])
def test_weights_it_refuses(name, cuda):
    """Weights whose fp64 sums are not exact, or not plain numbers, are the
    owner engine's."""
    import torch
    g = graphs.rmat(12, 16, seed=6)
    w = grid_weights(g.n, 8)
    if name == "wide":
        w[::2] *= np.float32(2.0 ** -40)
    else:
        w[5] = {"negative": -1.0, "infinite": np.inf, "nan": np.nan}[name]
    dg = api.DeviceCSR.from_host(g, cuda)
    W = torch.from_numpy(w).to(cuda)
    out, done = run(dg, W, api.ENGINE_ORIENTED, cuda)
    assert not done
    assert same(out, run(dg, W, api.ENGINE_OWNER, cuda)[0])


def test_default_route_replayed_in_a_graph(cuda):
    """From its size on the default call takes the oriented engine; captured
    with a workspace and replayed between eager calls it gives the same bits,
    edge-centric and vertex-centric."""
    import torch
    g = graphs.rmat(18, 16, seed=9)
    assert g.m >= 1 << 22
    dg = api.DeviceCSR.from_host(g, cuda)
    W = torch.from_numpy(grid_weights(g.n, 3)).to(cuda)
    want, _ = run(dg, W, api.ENGINE_OWNER, cuda)
    assert same(api.jaccard(dg, weights=W), want)
    assert same(api.jaccard(dg, weights=W, edge_centric=False), want)
    ws = torch.empty(api.workspace_size(g.n, g.m, True, True), dtype=torch.uint8, device=cuda)
    out = torch.empty(g.m, dtype=torch.float32, device=cuda)
    api.jaccard(dg, result=out, weights=W, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        api.jaccard(dg, result=out, weights=W, workspace=ws)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, want)
        assert same(api.jaccard(dg, weights=W), want)
    # a workspace of the owner engine's size is still enough
    small = torch.empty(96 << 20, dtype=torch.uint8, device=cuda)
    assert small.numel() < ws.numel()
    assert same(api.jaccard(dg, weights=W, workspace=small), want)
