"""The oriented engine's kernels for long rows at high ranks and for large |R|, on
graphs that it accepts: the counters in its workspace show that each had work.
Equal bit for bit with the owner engine; the smaller graphs with the oracle too."""
import numpy as np
import pytest

import oracle
from jaccard_amd import api, batch, graphs

pytestmark = pytest.mark.gpu

# counters of the engine's control words, one to 256 bytes
TASK16, TASK32, WAVE, RED_MID, RED_BIG = 9, 10, 11, 14, 15


def grid_weights(n, seed):
    return ((1 + np.random.default_rng(seed).integers(0, 1 << 24, n)) * 2.0 ** -24).astype(np.float32)


def layers(k, width, seed=5):
    """A clique of k vertices, each also tied to `width` others of its own, which
    pay for its part of the bit matrix: |R| up to k - 1."""
    a, b = np.triu_indices(k, 1)
    return graphs.from_edges(k + k * width, np.concatenate([a, np.repeat(np.arange(k), width)]),
                             np.concatenate([b, k + np.arange(k * width)]))


def circulant(n, reach):
    """Every vertex next to the `reach` ids on both sides, sorted CSR made
    directly: rows of 2 * reach entries at every rank."""
    d = np.concatenate([np.arange(-reach, 0), np.arange(1, reach + 1)])
    ind = np.sort((np.arange(n)[:, None] + d) % n, axis=1).astype(np.int32).reshape(-1)
    return graphs.CSRGraph(n, (np.arange(n + 1) * 2 * reach).astype(np.int32), ind)


def clique_at_high_ranks():
    """A batch whose last graph has a clique: |R| above what the 16-bit kernel
    holds, at ranks of the whole above what the 32-bit kernel's table does."""
    b = batch.rmat_batch([65536] * 5, [16.0] * 5, [1, 2, 3, 4, 5], False)
    u, g = b.union, layers(1500, 20)
    return graphs.CSRGraph(u.n + g.n, np.concatenate([u.offsets, u.offsets[-1] + g.offsets[1:]]).astype(np.int32),
                           np.concatenate([u.indices, g.indices + u.n]).astype(np.int32))


# name: (graph, members, counters that must not be 0)
GRAPHS = {
    "clique_1600": (lambda: layers(1600, 1010), 0, (TASK16, TASK32, RED_MID, RED_BIG)),
    "rows_of_512_past_65535": (lambda: circulant(70000, 256), 0, (TASK16, TASK32, WAVE)),
    "batch_clique_at_high_ranks": (clique_at_high_ranks, 1, (TASK16, WAVE, RED_BIG)),
}


def owner_bytes(n, m, weighted):
    """Workspace of the owner engine, which the oriented engine's follows; stated
    by workspace_size below the size from which that includes both."""
    def al(v):
        return (v + 255) // 256 * 256

    def lists(n, m):
        tasks = m // 896 + min(n, m // 2) + 1
        return al(8 * tasks) + al(4 * n) + al(4 * tasks)

    def total(n, m):
        head = api.workspace_size(1, 1, False, True) - lists(1, 1)
        return head + lists(n, m) + (al(4 * (n + 4)) + al(8 * n) + 256 if weighted else 0)

    assert total(70000, 2000000) == api.workspace_size(70000, 2000000, weighted, True)
    return total(n, m)


@pytest.mark.parametrize("name", list(GRAPHS))
def test_long_rows(name, cuda):
    import torch
    make, members, busy = GRAPHS[name]
    g = make()
    dg = api.DeviceCSR.from_host(g, cuda)
    for weighted in (False, True):
        W = torch.from_numpy(grid_weights(g.n, 7)).to(cuda) if weighted else None
        need = owner_bytes(g.n, g.m, weighted)
        ws = torch.full((need + 48 * g.m + 256 * g.n + (1 << 20),), 0xA5, dtype=torch.uint8, device=cuda)
        print(f"[gpu] long rows {name} weighted={weighted} n={g.n} m={g.m}", flush=True)
        out = api.jaccard(dg, weights=W, workspace=ws, tuning=dict(engine=api.ENGINE_ORIENTED, members=members))
        ctl = ws[need:need + 16 * 256].view(torch.int32).cpu().numpy()
        assert ctl[1] == 1, "delivered"
        assert all(ctl[64 * k] > 0 for k in busy), [int(ctl[64 * k]) for k in busy]
        own = api.jaccard(dg, weights=W, tuning=dict(engine=api.ENGINE_OWNER))
        assert torch.equal(out.view(torch.int32), own.view(torch.int32))
        if g.m < 8 << 20:
            e = np.random.default_rng(1).choice(g.m, 20000, replace=False)
            rows = np.repeat(np.arange(g.n), np.diff(g.offsets))
            got = out.cpu().numpy()[e]
            if weighted:
                ref = oracle.pairs_weighted_f64(g, W.cpu().numpy().astype(np.float64), rows[e], g.indices[e])
                assert np.all(np.abs(got - ref) <= 1e-6 * np.abs(ref))
            else:
                ref = oracle.pairs_unweighted(g, rows[e], g.indices[e])
                assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        del ws
