"""Weighted pair lists by every way to the row sums (per pair, of all rows, as a
sample says) and both kinds of pairs in one workgroup: short rows by a wave
each, others cut into units. Bit for bit the same coefficients either way, and
as the coefficients of the stored edges; sums are exact in double-double."""
import numpy as np
import pytest

from jaccard_amd import api, graphs

pytestmark = pytest.mark.gpu

# name: graph; the sums' way at 1000, 20000 and 70000 pairs: per pair, all or per pair, all or asked
GRAPHS = {
    "skewed": lambda: graphs.rmat(17, 16, seed=3, weighted=True),
    "hubs": lambda: hubs(),
    "sparse": lambda: graphs.from_edges(400000, *np.random.default_rng(1).integers(0, 400000, (2, 300000))),
    "rows_of_512": lambda: ring(3000, 256),
    "rows_of_514": lambda: ring(3000, 257),
}


def hubs():
    """Three vertices next to all of 60000, which have random edges as well."""
    rng = np.random.default_rng(2)
    leaves = np.arange(3, 60003)
    return graphs.from_edges(60003, np.concatenate([np.repeat(np.arange(3), leaves.size), rng.integers(3, 60003, 90000)]),
                             np.concatenate([np.tile(leaves, 3), rng.integers(3, 60003, 90000)]))


def ring(n, reach):
    i = np.repeat(np.arange(n), reach)
    return graphs.from_edges(n, i, (i + np.tile(np.arange(1, reach + 1), n)) % n)


@pytest.mark.parametrize("name", list(GRAPHS))
def test_pairs_equal_edges(name, cuda):
    import torch
    g = GRAPHS[name]()
    dg = api.DeviceCSR.from_host(g, cuda)
    w = ((1 + np.random.default_rng(5).integers(0, 1 << 24, g.n)) * 2.0 ** -24).astype(np.float32)
    W = torch.from_numpy(w).to(cuda)
    every = {False: api.jaccard(dg), True: api.jaccard(dg, weights=W)}
    rows = np.repeat(np.arange(g.n, dtype=np.int32), np.diff(g.offsets))
    rng = np.random.default_rng(6)
    for count in (1, 7, 1000, 20000, 70000):
        e = rng.integers(0, g.m, count)
        first, second = rows[e].copy(), g.indices[e].copy()
        bad = rng.random(count) < 0.01
        first[bad] = np.where(rng.random(bad.sum()) < 0.5, -1, g.n)
        f, s = torch.from_numpy(first).to(cuda), torch.from_numpy(second).to(cuda)
        at = torch.from_numpy(e).to(cuda)
        miss = torch.from_numpy(bad).to(cuda)
        print(f"[gpu] pair sums {name} n={g.n} m={g.m} pairs={count}", flush=True)
        for weighted in (False, True):
            out = api.jaccard_list(dg, f, s, weights=W if weighted else None)
            assert torch.equal(torch.isnan(out), miss)
            assert torch.equal(out[~miss].view(torch.int32), every[weighted][at][~miss].view(torch.int32)), weighted
