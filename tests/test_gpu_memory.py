"""Workspaces of calls without one of their own: the same results from several
threads and streams at once, under capture, and after what is kept between
calls was given back; and no more kept than the header says.
"""
import threading

import numpy as np
import pytest

from jaccard_amd import api, graphs

pytestmark = pytest.mark.gpu


def test_threads_streams_capture_and_release(cuda):
    import torch
    g = graphs.rmat(16, 24)
    dg = api.DeviceCSR.from_host(g, cuda)
    want = api.jaccard(dg, edge_centric=False)
    torch.cuda.synchronize()
    outs = [[torch.empty(g.m, device=cuda) for _ in range(4)] for _ in range(4)]
    torch.cuda.synchronize()
    print(f"[gpu] workspaces n={g.n} m={g.m}", flush=True)

    def work(mine):
        stream = torch.cuda.Stream(device=cuda)
        for k, out in enumerate(mine):
            api.jaccard(dg, result=out, edge_centric=False, stream=stream)
            if k == 1:
                api.release_workspaces()
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(o,)) for o in outs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for mine in outs:
        for out in mine:
            assert torch.equal(out.view(torch.int32), want.view(torch.int32))

    out = torch.zeros(g.m, device=cuda)
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream(device=cuda)
    with torch.cuda.graph(graph, stream=stream):
        api.jaccard(dg, result=out, edge_centric=False, stream=stream)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
        api.jaccard(dg, edge_centric=False)


def test_kept_memory_is_bounded(cuda):
    import torch
    n, e = 1 << 20, 40 << 20  # 80M directed entries: 1.9 GB of temporaries and more
    gen = torch.Generator(device=cuda).manual_seed(1)
    s, d = (torch.randint(0, n, (e,), generator=gen, device=cuda, dtype=torch.int32) for _ in range(2))
    w = torch.rand(e, generator=gen, device=cuda)
    torch.cuda.synchronize()
    api.release_workspaces()
    free0 = torch.cuda.mem_get_info()[0]
    print(f"[gpu] kept memory, ingest of {e} draws", flush=True)
    g = api.csr_from_edges(n, s, d, w)
    m = g.m
    del g
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert m > 79_000_000
    slack = 64 << 20  # blocks are whole pages of the pool
    assert free0 - torch.cuda.mem_get_info()[0] <= (2 << 30) + slack
    api.release_workspaces()
    assert free0 - torch.cuda.mem_get_info()[0] <= slack
