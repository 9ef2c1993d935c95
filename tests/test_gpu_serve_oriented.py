"""Serving batches large enough for the oriented engine: the copy of the
requested graphs (all small enough to be ranked by themselves, or not), a
budget that has room for it or has not, a request set that is not the whole
arena, and graphs of even degree that the engine turns down. The same bits as
one call per graph in every case."""
import numpy as np
import pytest

from jaccard_amd import api, graphs, serve

pytestmark = pytest.mark.gpu


def ring(n, k):
    i = np.repeat(np.arange(n), k)
    return graphs.from_edges(n, i, (i + 1 + np.tile(np.arange(k), n)) % n)


@pytest.fixture(scope="module")
def sets():
    def r(scale, ef, seed):
        return graphs.rmat(scale, ef, seed=seed, weighted=True)

    rng = np.random.default_rng(2)
    even = ring(60000, 60)
    even.weights = (rng.integers(1, 64, even.m) / 64).astype(np.float32)
    return {"small": [r(12, 16, 1), r(16, 32, 2), r(15, 40, 3), r(16, 24, 4)],
            "large": [r(17, 28, 5), r(13, 8, 6), r(16, 16, 7)],
            "even": [even, r(10, 8, 8)]}


@pytest.mark.parametrize("weighted", [True, False])
@pytest.mark.parametrize("name,budget", [("small", 1 << 30), ("large", 1 << 30), ("even", 1 << 30), ("small", 32 << 20)])
def test_large_batches(name, budget, weighted, sets, cuda):
    import torch
    gs = sets[name]
    dev = serve.upload(gs, cuda, weighted=weighted)
    srv = serve.Server(gs, cuda, weighted=weighted, slots=2, hbm_budget_bytes=budget, device_graphs=dev)
    want = []
    for dg, W in dev:
        W = W if weighted else None
        want.append(api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER)))
    rng = np.random.default_rng(1)
    print(f"[gpu] serve large batches {name} budget={budget} weighted={weighted}", flush=True)
    for which in (range(len(gs)), [1], [len(gs) - 1, 0]):
        reqs = [serve.Request(g, serve.REQ_FULL, 0.0) for g in which]
        g = list(which)[0]
        reqs.append(serve.Request(g, serve.REQ_PAIRS, 0.0, rng.integers(0, gs[g].n, 100).astype(np.int32),
                                  rng.integers(0, gs[g].n, 100).astype(np.int32)))
        reqs += [serve.Request(g, serve.REQ_FULL, 0.0) for g in which]  # a second batch
        res = serve.result_buffers(gs, reqs, cuda)
        st, info = srv.run(reqs, res)
        assert (st["status"] == 0).all()
        assert info["peak_budget_bytes"] <= budget
        for q, out in zip(reqs, res):
            if q.kind == serve.REQ_FULL:
                assert torch.equal(out.view(torch.int32), want[q.graph].view(torch.int32)), (name, q.graph)
        edges = sum(gs[g].m for g in which)
        if budget == 1 << 30 and edges >= 6 << 20:  # the copy was made
            assert info["peak_budget_bytes"] > 30 * edges
        if budget < 1 << 30:
            assert info["peak_budget_bytes"] <= budget
    srv.close()
