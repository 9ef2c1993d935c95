"""A whole-graph request whose copy has to wait for memory is not held back by
smaller ones that keep coming: it is served after at most as many batches as
there are slots."""
import numpy as np
import pytest

from jaccard_amd import api, graphs, serve

pytestmark = pytest.mark.gpu


def test_large_request_among_smaller_ones(cuda):
    import torch
    gs = [graphs.rmat(17, 16, seed=s, weighted=True) for s in range(1, 9)] + [graphs.rmat(19, 16, seed=9, weighted=True)]
    large = len(gs) - 1
    assert min(g.m for g in gs) >= 3 << 20
    # one smaller graph's copy leaves too little for the large one's
    s = serve.Server(gs, cuda, slots=4, hbm_budget_bytes=900 << 20, max_batch_edges=3 << 20)
    order = [0, large] + [i % large for i in range(1, 40)]
    reqs = [serve.Request(g, serve.REQ_FULL, 0.0) for g in order]
    res = serve.result_buffers(gs, reqs, cuda)
    print(f"[gpu] serve order m={gs[large].m}", flush=True)
    st, info = s.run(reqs, res)
    s.close()
    assert (st["status"] == 0).all()
    assert info["batches"] >= 40
    assert st["batch"][1] <= 1 + 4
    for g, out in zip(order, res):
        own = api.jaccard(s.dev[g][0], weights=s.dev[g][1], tuning=dict(engine=api.ENGINE_OWNER))
        assert torch.equal(out.view(torch.int32), own.view(torch.int32))
