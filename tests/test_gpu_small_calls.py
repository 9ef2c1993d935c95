"""The one-launch paths for small graphs: the kernel that holds the whole CSR in
LDS up to its last byte and just past it, one-launch row sums around their row
classes, the one-pass schedule, against the oracle. Any CSR is accepted:
asymmetric ones and self loops too.

Unweighted results are bit-exact; weighted ones carry one fp32 rounding of
sums that are exact in double-double (the repository's 1e-6 bounds it).
"""
import numpy as np
import pytest

import oracle
from jaccard_amd import api, graphs

import cases

pytestmark = pytest.mark.gpu

LDS = 150 * 1024


def ring(n, m):
    """n vertices and exactly m stored entries (m even, at least 2): a path's
    first edges, then chords."""
    e = m // 2
    i = np.arange(e)
    step = 1 + i // n
    return graphs.from_edges(n, i % n, (i % n + step) % n)


def directed(n, seed):
    rng = np.random.default_rng(seed)
    return graphs.from_edges(n, rng.integers(0, n, 6 * n), rng.integers(0, n, 6 * n), symmetrize=False)


def with_loop(g):
    rows = np.repeat(np.arange(g.n), np.diff(g.offsets))
    rows, cols = np.append(rows, g.n // 2), np.append(g.indices, g.n // 2)
    order = np.lexsort((cols, rows))
    off = np.zeros(g.n + 1, np.int32)
    np.add.at(off, rows + 1, 1)
    return graphs.CSRGraph(g.n, np.cumsum(off).astype(np.int32), cols[order].astype(np.int32))


# entries that fill the LDS exactly beside n = 1501 vertices, unweighted and weighted
FIT_U = LDS // 4 - 1502
FIT_W = (LDS - 12 * 1501) // 4 - 1502
GRAPHS = {
    "k2": lambda: cases.complete(2),
    "path": lambda: cases.path(19),
    "star_1600": lambda: cases.star(1600),
    "rmat9": lambda: graphs.rmat(9, 8, seed=5),
    "fits_unweighted": lambda: ring(1501, FIT_U - FIT_U % 2),
    "past_unweighted": lambda: ring(1501, FIT_U - FIT_U % 2 + 2),
    "fits_weighted": lambda: ring(1501, FIT_W - FIT_W % 2),
    "past_weighted": lambda: ring(1501, FIT_W - FIT_W % 2 + 2),
    "directed": lambda: directed(400, 2),
    "directed_past": lambda: directed(9000, 3),
    "self_loop": lambda: with_loop(graphs.rmat(8, 8, seed=2)),
    "self_loop_past": lambda: with_loop(graphs.rmat(13, 16, seed=2)),
    "rows_64_65_1024_1025": lambda: graphs.from_edges(
        4000, np.repeat([0, 1, 2, 3], [64, 65, 1024, 1025]),
        np.concatenate([np.arange(10, 74), np.arange(10, 75), np.arange(100, 1124), np.arange(100, 1125)])),
    "one_pass_schedule": lambda: graphs.rmat(15, 16, seed=8),
}


@pytest.mark.parametrize("name", list(GRAPHS))
def test_small_graphs(name, cuda):
    import torch
    g = GRAPHS[name]()
    print(f"[gpu] small {name} n={g.n} m={g.m}", flush=True)
    w = ((1 + np.random.default_rng(3).integers(0, 1 << 24, g.n)) * 2.0 ** -20).astype(np.float32)
    ew = ((1 + np.random.default_rng(4).integers(0, 1 << 24, g.m)) * 2.0 ** -24).astype(np.float32)
    dg = api.DeviceCSR(g.n, *(torch.from_numpy(x).to(cuda) for x in (g.offsets, g.indices, ew)))
    ref = oracle.ec_unweighted(g)
    for ec in (True, False):
        out = api.jaccard(dg, edge_centric=ec).cpu().numpy()
        assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    sums = np.zeros(g.n)
    np.add.at(sums, np.repeat(np.arange(g.n), np.diff(g.offsets)), ew.astype(np.float64))
    got = api.vertex_weights(dg).cpu().numpy()
    assert np.array_equal(got, sums.astype(np.float32))  # 24-bit multiples: exact, then one rounding
    W = torch.from_numpy(w).to(cuda)
    refw = oracle.weighted_f64(g, w.astype(np.float64))
    outs = [api.jaccard(dg, weights=W), api.jaccard(dg, weights=W, edge_centric=False),
            api.jaccard_noalloc(dg, weights=W), api.jaccard(dg, weights=W, tuning=dict(small_max=128))]
    for o in outs:
        assert torch.equal(o.view(torch.int32), outs[0].view(torch.int32))
        o = o.cpu().numpy().astype(np.float64)
        assert np.all(np.abs(o - refw) <= 1e-6 * np.abs(refw))


@pytest.mark.parametrize("n", [(2 << 20) - 1, 2 << 20, (2 << 20) + 1])
def test_row_sums_of_many_rows(n, cuda):
    """Both sides of the number of rows that row sums take in one launch: a
    row of 70,000 entries, one of 1,500, short ones, empty ones at both ends."""
    import torch
    rng = np.random.default_rng(n)
    deg = np.zeros(n, np.int64)
    deg[rng.integers(10, n - 10, 50000)] = rng.integers(1, 40, 50000)
    deg[n // 2], deg[n // 3] = 70000, 1500
    off = np.concatenate([[0], np.cumsum(deg)])
    ind = rng.integers(0, n, off[-1]).astype(np.int32)
    w = rng.random(off[-1]).astype(np.float32)
    v = rng.random(n).astype(np.float32)
    print(f"[gpu] row sums n={n} m={off[-1]}", flush=True)
    dg = api.DeviceCSR(n, torch.from_numpy(off.astype(np.int32)).to(cuda), torch.from_numpy(ind).to(cuda),
                       torch.from_numpy(w).to(cuda))
    live = np.flatnonzero(deg)

    def sums(x):
        s = np.zeros(n)
        s[live] = np.add.reduceat(x.astype(np.float64), off[live])
        return s

    np.testing.assert_allclose(api.vertex_weights(dg).cpu().numpy(), sums(w), rtol=1e-6, atol=0)
    out = torch.empty(n, device=cuda)
    api.rowsum(dg, out, v=torch.from_numpy(v).to(cuda))
    np.testing.assert_allclose(out.cpu().numpy(), sums(v[ind]), rtol=1e-6, atol=0)
