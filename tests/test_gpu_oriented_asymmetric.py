"""Graphs that are symmetric but for a few entries, through the oriented
engine: it has to find out and leave the result to the owner engine.

Two stored entries are missing, one on either side of the orientation, so the
entry count alone does not show it, and a sample of 1024 entries misses them.
The workspace holds old or arbitrary bytes, as a recycled one does. Results of
both engines are equal bit for bit: counts are integers, and the weights are
multiples of 2^-24 whose sums are exact.
"""
import numpy as np
import pytest

import oracle
from jaccard_amd import api, graphs

pytestmark = pytest.mark.gpu


def grid_weights(n, seed):
    return ((1 + np.random.default_rng(seed).integers(0, 1 << 24, n)) * 2.0 ** -24).astype(np.float32)


def without(g, entries):
    """g less the stored entries (u, v)."""
    drop = [int(g.offsets[u] + np.searchsorted(g.indices[g.offsets[u]:g.offsets[u + 1]], v)) for u, v in entries]
    assert all(g.indices[k] == v for k, (_, v) in zip(drop, entries))
    off = g.offsets.astype(np.int64).copy()
    for u, _ in entries:
        off[u + 1:] -= 1
    return graphs.CSRGraph(g.n, off.astype(np.int32), np.delete(g.indices, drop).astype(np.int32))


def balanced(g, degree):
    """g less (x, v), x of the given degree and v above it, and less (h, l), h
    the vertex of most neighbours and l one of its lesser ones. With degree 1
    the row of x is then empty, and v still names it."""
    deg = np.diff(g.offsets)
    row = lambda u: g.indices[g.offsets[u]:g.offsets[u + 1]]
    h = int(np.argmax(deg))
    x = next(int(u) for u in np.flatnonzero(deg == degree) if h not in row(u) and deg[row(u)[0]] > 4 * degree + 16)
    v = int(row(x)[0])
    l = next(int(u) for u in row(h) if 4 <= deg[u] < deg[h] // 4 and u != v)
    a = without(g, [(x, v), (h, l)])
    d = np.diff(a.offsets)
    assert d[x] == degree - 1 and d[v] > d[x] and d[h] > 2 * d[l] and a.m == g.m - 2
    return a


def looped(g, shortest):
    """g with a self loop at every vertex of at least `shortest` neighbours: a
    loop is its own mirror, so only the rows themselves show it."""
    deg = np.diff(g.offsets)
    rows = np.repeat(np.arange(g.n), deg)
    at = np.flatnonzero(deg >= shortest)
    assert at.size > 8
    key = np.sort(np.concatenate([rows.astype(np.int64) * g.n + g.indices, at * (g.n + 1)]))
    off = np.zeros(g.n + 1, np.int32)
    off[1:] = np.cumsum(np.bincount(key // g.n, minlength=g.n))
    return graphs.CSRGraph(g.n, off, (key % g.n).astype(np.int32))


def call(dg, W, ws, device):
    """The oriented engine's call over the bytes of ws: result, delivered."""
    need = api.workspace_size(dg.n, dg.m, W is not None, True)
    assert dg.m < 3 << 20 and ws.numel() >= need + 64 * dg.m + 256 * dg.n
    out = api.jaccard(dg, weights=W, workspace=ws, tuning=dict(engine=api.ENGINE_ORIENTED))
    return out, int(ws[need + 4:need + 8].view(__import__("torch").int32)) == 1


def same(a, b):
    import torch
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("shortest", [2, 65, 1025])
def test_self_loops(shortest, cuda):
    """In rows of every class that orient takes by itself: while some
    workgroups find them, others of the launch begin."""
    import torch
    a = looped(graphs.rmat(15, 32, seed=5), shortest)
    dg = api.DeviceCSR.from_host(a, cuda)
    for weighted in (False, True):
        W = torch.from_numpy(grid_weights(a.n, 7)).to(cuda) if weighted else None
        ws = torch.full((api.workspace_size(a.n, a.m, weighted, True) + 64 * a.m + 256 * a.n + (1 << 20),), 0xA5,
                        dtype=torch.uint8, device=cuda)
        print(f"[gpu] self loops from {shortest} weighted={weighted} n={a.n} m={a.m}", flush=True)
        out, done = call(dg, W, ws, cuda)
        assert not done and same(out, api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER)))


@pytest.mark.parametrize("degree", [1, 3])
def test_missing_mirrors_that_balance(degree, cuda):
    import torch
    g = graphs.rmat(14, 16, seed=2)
    a = balanced(g, degree)
    dg, whole = (api.DeviceCSR.from_host(x, cuda) for x in (a, g))
    for weighted in (False, True):
        W = torch.from_numpy(grid_weights(g.n, 7)).to(cuda) if weighted else None
        own = api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER))
        if not weighted:
            assert np.array_equal(own.cpu().numpy().view(np.uint32), oracle.ec_unweighted(a).view(np.uint32))
        ws = torch.full((api.workspace_size(g.n, g.m, weighted, True) + 64 * g.m + 256 * g.n + (1 << 20),), 0xA5,
                        dtype=torch.uint8, device=cuda)
        print(f"[gpu] asymmetric degree={degree} weighted={weighted} n={a.n} m={a.m}", flush=True)
        out, done = call(dg, W, ws, cuda)
        assert not done and same(out, own)
        _, done = call(whole, W, ws, cuda)
        assert done
        out, done = call(dg, W, ws, cuda)
        assert not done and same(out, own)


def test_default_route(cuda):
    """The same from the size on at which the plain call tries the engine."""
    import torch
    g = graphs.rmat(18, 16, seed=9)
    a = balanced(g, 1)
    assert a.m >= 3 << 20
    W = torch.from_numpy(grid_weights(g.n, 3)).to(cuda)
    dg, whole = (api.DeviceCSR.from_host(x, cuda) for x in (a, g))
    own = api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER))
    ws = torch.full((api.workspace_size(g.n, g.m, True, True),), 0x5A, dtype=torch.uint8, device=cuda)
    print(f"[gpu] asymmetric default n={a.n} m={a.m}", flush=True)
    assert same(api.jaccard(dg, weights=W, workspace=ws), own)
    api.jaccard(whole, weights=W, workspace=ws)
    assert same(api.jaccard(dg, weights=W, workspace=ws), own)
    assert same(api.jaccard(dg, weights=W), own)


def test_entry_before_the_first_part(cuda):
    """A batch that begins with vertices without neighbours, and an entry that
    names one of them all the same; another is missing, so the counts agree."""
    import torch
    from jaccard_amd import batch
    pad = 37
    u = batch.rmat_batch([700, 9001, 4096], [9.0, 12.0, 16.0], [1, 2, 3], False).union
    g = graphs.CSRGraph(u.n + pad, np.concatenate([np.zeros(pad, np.int32), u.offsets]).astype(np.int32),
                        (u.indices + pad).astype(np.int32))
    deg = np.diff(g.offsets)
    h = int(np.argmax(deg))
    a = without(g, [(h, next(int(l) for l in g.indices[g.offsets[h]:g.offsets[h + 1]] if 4 <= deg[l] < deg[h] // 4))])
    v = int(np.flatnonzero(deg > 40)[0])  # in the first part: 3 ranks after it
    off = a.offsets.copy()
    off[v + 1:] += 1
    a = graphs.CSRGraph(a.n, off, np.insert(a.indices, a.offsets[v], 3).astype(np.int32))
    assert a.m == g.m
    dg = api.DeviceCSR.from_host(a, cuda)
    for weighted in (False, True):
        W = torch.from_numpy(grid_weights(a.n, 7)).to(cuda) if weighted else None
        need = api.workspace_size(a.n, a.m, weighted, True)
        ws = torch.full((need + 64 * a.m + 256 * a.n + (1 << 20),), 0x5A, dtype=torch.uint8, device=cuda)
        print(f"[gpu] asymmetric members weighted={weighted} n={a.n} m={a.m}", flush=True)
        out = api.jaccard(dg, weights=W, workspace=ws, tuning=dict(engine=api.ENGINE_ORIENTED, members=1))
        assert int(ws[need + 4:need + 8].view(torch.int32)) == 0
        assert same(out, api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER)))
