"""Workspaces of calls without one of their own are memory that stays mapped:
graphs of any size on a stream use one block, the largest call's, also when
every call is waited for; a stream that finds it in use takes another."""
import threading

import numpy as np
import pytest

from jaccard_amd import api, graphs

pytestmark = pytest.mark.gpu


def uniform(n, m, cuda):
    """About m stored entries of a symmetric random graph, built on the device."""
    import torch
    gen = torch.Generator(device=cuda).manual_seed(1)
    a, b = (torch.randint(0, n, (m // 2,), generator=gen, device=cuda) for _ in range(2))
    k = torch.unique(torch.cat([a * n + b, b * n + a]))
    k = k[k // n != k % n]
    off = torch.zeros(n + 1, dtype=torch.int64, device=cuda)
    off[1:] = torch.cumsum(torch.bincount(k // n, minlength=n), 0)
    return api.DeviceCSR(n, off.int().contiguous(), (k % n).int().contiguous())


def free(torch):
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def test_one_block_serves_all_sizes(cuda):
    import torch
    sizes = [(1 << 21, 80 << 20), (1 << 20, 40 << 20), (1 << 17, 10 << 20), (1 << 16, 2 << 20)]
    gs = [uniform(n, m, cuda) for n, m in sizes]
    outs = [torch.empty(g.m, device=cuda) for g in gs]
    need = api.workspace_size(gs[0].n, gs[0].m, False, True)
    assert (2 << 30) < need < (4 << 30)  # more than a little memory, and not all that is kept
    api.release_workspaces()
    free0 = free(torch)
    print(f"[gpu] workspace of {need} bytes", flush=True)
    api.jaccard(gs[0], result=outs[0])
    kept = free0 - free(torch)
    slack = 64 << 20
    assert need - slack <= kept <= need + slack
    want = [o.clone() for o in outs[:1]]
    base = free(torch)
    for k in (1, 2, 0, 3, 1, 2, 0):
        api.jaccard(gs[k], result=outs[k])
        torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int32), want[0].view(torch.int32))
    assert abs(base - free(torch)) <= slack
    # a smaller graph first: the block grows, and is not added to
    api.release_workspaces()
    del want
    base = free(torch)
    for k in (3, 2, 1, 0):
        api.jaccard(gs[k], result=outs[k])
        torch.cuda.synchronize()
    assert base - free(torch) <= need + need // 4 + slack
    api.release_workspaces()
    assert base - free(torch) <= slack


def test_streams_that_overlap(cuda):
    """Each stream's calls wait for the block's last work and for nothing else;
    streams come and go, and their handles with them."""
    import torch
    g = graphs.rmat(17, 24, weighted=True)
    dg = api.DeviceCSR.from_host(g, cuda)
    W = api.vertex_weights(dg)
    want = api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER))
    torch.cuda.synchronize()
    print(f"[gpu] streams n={g.n} m={g.m}", flush=True)
    for _ in range(4):
        streams = [torch.cuda.Stream(device=cuda) for _ in range(6)]
        outs = [torch.zeros(g.m, device=cuda) for _ in range(12)]
        torch.cuda.synchronize()
        for k, out in enumerate(outs):
            api.jaccard(dg, result=out, weights=W, stream=streams[k % 6])
        del streams
        torch.cuda.synchronize()
        for out in outs:
            assert torch.equal(out.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("capture_first", [True, False])
def test_calls_while_another_thread_captures(capture_first, cuda):
    """Calls that take memory beside a capture, larger ones each time: neither they
    nor any replay of the graph, with calls in between, may come out different."""
    import torch
    g = graphs.rmat(13, 16)
    dg = api.DeviceCSR.from_host(g, cuda)
    want = api.jaccard(dg)
    torch.cuda.synchronize()
    for scale in (13, 14, 15, 16, 17, 18):
        big = api.DeviceCSR.from_host(graphs.rmat(scale, 16), cuda)
        a, b = torch.zeros(g.m, device=cuda), torch.zeros(big.m, device=cuda)
        side, main = torch.cuda.Stream(device=cuda), torch.cuda.Stream(device=cuda)
        torch.cuda.synchronize()
        graph, errors = torch.cuda.CUDAGraph(), []

        def work():
            try:
                for _ in range(3):
                    api.jaccard(big, result=b, stream=side)
            except Exception as e:  # noqa: BLE001
                errors.append(e)

        print(f"[gpu] calls beside a capture, 2^{scale} vertices", flush=True)
        with torch.cuda.graph(graph, stream=main):
            if capture_first:
                api.jaccard(dg, result=a, stream=main)
            t = threading.Thread(target=work)
            t.start()
            t.join()
            if not capture_first:
                api.jaccard(dg, result=a, stream=main)
        side.synchronize()
        assert not errors
        own = api.jaccard(big, tuning=dict(engine=api.ENGINE_OWNER))
        assert torch.equal(b.view(torch.int32), own.view(torch.int32))
        for _ in range(4):
            a.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(a.view(torch.int32), want.view(torch.int32))
            api.jaccard(big, result=b)
            torch.cuda.synchronize()
            assert torch.equal(b.view(torch.int32), own.view(torch.int32))
