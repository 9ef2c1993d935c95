"""A union is announced as one of small graphs only where each of them is as small
as that says (at most 65536 vertices)."""
import numpy as np
import pytest

from jaccard_amd import api, batch


def test_only_small_graphs_are_members():
    sizes = {(700, 65536): 1, (700, 65537): 0, (100003,): 0, (2,): 1}
    for ns, want in sizes.items():
        b = batch.rmat_batch(list(ns), [2.0] * len(ns), list(range(1, len(ns) + 1)), False)
        assert batch._members(b) == want, ns


@pytest.mark.gpu
def test_batch_with_a_large_graph(cuda):
    import torch
    ns, efs = [100003, 4096, 65536], [16.0, 16.0, 16.0]
    bs = [batch.rmat_batch(ns, efs, [1, 2, 3], weighted) for weighted in (False, True)]
    r = batch.BatchRunner(bs)
    r.select()
    r.capture()
    print(f"[gpu] batch with a large graph m={[b.union.m for b in bs]}", flush=True)
    for _ in range(2):
        r.replay()
        torch.cuda.synchronize()
        for k, b in enumerate(bs):
            it = r.items[k]
            assert it["members"] == 0
            own = api.jaccard(it["dg"], weights=it["W"], tuning=dict(engine=api.ENGINE_OWNER))
            assert torch.equal(own.view(torch.int32), it["out"].view(torch.int32))
