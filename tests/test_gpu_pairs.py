"""Pair lists whose rows end at and around the pair kernel's units: 64 entries
of the longer row, 64 and 128 of the shorter one, 1024 of a row sum, more pairs
than workgroups, and both ways to the row sums, against the oracle.

Unweighted results are bit-exact; weighted ones carry one fp32 rounding of
sums that are exact in double-double (the repository's 1e-6 bounds it).
"""
import numpy as np
import pytest

import oracle
from jaccard_amd import api, graphs

pytestmark = pytest.mark.gpu

LENS = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 257, 1023, 1024, 1025, 2049, 5000]


@pytest.fixture(scope="module")
def rows():
    """Directed rows of the given lengths over 6000 ids, some of them nested."""
    rng = np.random.default_rng(3)
    n = 6000
    src, dst = [], []
    for u, d in enumerate(LENS):
        src += [u] * d
        dst += (200 + rng.choice(n - 200, size=d, replace=False)).tolist()
    for u, d in enumerate(LENS):
        src += [100 + u] * d
        dst += list(range(n - d, n))  # a run at the end of the ids
    return graphs.from_edges(n, np.array(src), np.array(dst), symmetrize=False)


@pytest.mark.parametrize("count", [1, 5, 1024, 20000])
def test_pairs_around_units(cuda, rows, count):
    import torch
    g = rows
    assert all(np.diff(g.offsets)[u] == d for u, d in enumerate(LENS))
    ids = np.concatenate([np.arange(len(LENS)), 100 + np.arange(len(LENS))])
    every = np.stack(np.meshgrid(ids, ids), -1).reshape(-1, 2)  # 1024 pairs
    rng = np.random.default_rng(count)
    every = every[rng.permutation(len(every))]
    first, second = np.resize(every, (count, 2)).astype(np.int32).T.copy()
    print(f"[gpu] pairs count={count}", flush=True)
    dg = api.DeviceCSR.from_host(g, cuda)
    f, s = torch.from_numpy(first).to(cuda), torch.from_numpy(second).to(cuda)
    k = min(count, len(every))
    ref = np.resize(oracle.pairs_unweighted(g, first[:k], second[:k]), count)
    out = api.jaccard_list(dg, f, s).cpu().numpy()
    assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    v = (rng.random(g.n) + 0.1).astype(np.float32)
    w = torch.from_numpy(v).to(cuda)
    refw = np.resize(oracle.pairs_weighted_f64(g, v.astype(np.float64), first[:k], second[:k]), count)
    outw = api.jaccard_list(dg, f, s, weights=w).cpu().numpy()
    assert np.array_equal(np.isnan(outw), np.isnan(refw))
    np.testing.assert_allclose(outw, refw, rtol=1e-6, atol=0)
    # the kernel-level form adds to what is there
    work = torch.empty(g.n, device=cuda)
    api.rowsum(dg, work, v=w)
    wi, ws = torch.full((count,), 2.0, device=cuda), torch.empty(count, device=cuda)
    api.intersect_pairs(dg, f, s, work, wi, ws, v=w)
    deg = np.diff(g.offsets)
    both = work.cpu().numpy()
    assert np.array_equal(ws.cpu().numpy(), both[first] + both[second])
    rowset = [g.indices[g.offsets[u]:g.offsets[u + 1]] for u in range(g.n)]
    for i in range(0, k, 37):
        common = np.intersect1d(rowset[first[i]], rowset[second[i]])
        want = np.float32(2.0) + np.float32(v[common].astype(np.float64).sum())
        assert wi[i].item() == pytest.approx(float(want), rel=3e-7)
    assert deg.max() == 5000
