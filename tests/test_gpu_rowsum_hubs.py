"""Row sums of graphs with rows long enough for a workgroup of their own: next to
each other, first, last, of the limit's length and one either side of it, among empty
rows. Sums are exact in double-double, rounded once, so fp32 sums equal fp64
ones of the same order-free exact sum rounded to fp32."""
import numpy as np
import pytest

from jaccard_amd import api

pytestmark = pytest.mark.gpu

HUB = 32768

# row lengths, rows in between are empty or short
ROWS = {
    "limit": [HUB - 1, HUB, HUB + 1, 0, 3],
    "neighbours": [HUB + 1] * 7 + [2 * HUB, 2 * HUB + 1, 3 * HUB - 1],
    "first_and_last": [100000] + [0, 1, 5, 64, 65, 1024, 1025] * 300 + [65536],
    "only": [200000],
    "none": [HUB] * 4 + [1] * 50000,
    "ends_on_a_stretch": [HUB, HUB, 2 * HUB, 4 * HUB, 1],
}


@pytest.mark.parametrize("name", list(ROWS))
def test_row_sums(name, cuda):
    import torch
    lens = np.array(ROWS[name])
    n = max(int(lens.max()) + 1, HUB + 5, lens.size)
    d = np.zeros(n, np.int64)
    d[np.sort(np.random.default_rng(1).choice(n, lens.size, replace=False)) if name != "first_and_last"
      else np.r_[0, 1 + np.arange(lens.size - 2) * 7, n - 1]] = lens
    off = np.zeros(n + 1, np.int32)
    off[1:] = np.cumsum(d)
    m = int(off[-1])
    rng = np.random.default_rng(2)
    ind = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in d if k]).astype(np.int32)
    v = ((1 + rng.integers(0, 1 << 24, n)) * 2.0 ** -24).astype(np.float32)
    w = ((1 + rng.integers(0, 1 << 24, m)) * 2.0 ** -24).astype(np.float32)
    rows = np.repeat(np.arange(n), d)
    print(f"[gpu] hub rows {name} n={n} m={m} longest={d.max()}", flush=True)
    g = api.DeviceCSR(n, *(torch.from_numpy(x).to(cuda) for x in (off, ind, w)))
    # below 2^53 units of 2^-24: bincount's fp64 sums are exact
    got = api.vertex_weights(g).cpu().numpy()
    assert np.array_equal(got, np.bincount(rows, w.astype(np.float64), n).astype(np.float32))
    out = torch.full((n,), -1.0, device=cuda)
    api.rowsum(g, out, v=torch.from_numpy(v).to(cuda))
    assert np.array_equal(out.cpu().numpy(), np.bincount(rows, v[ind].astype(np.float64), n).astype(np.float32))


@pytest.mark.parametrize("wide", [False, True])
def test_coefficients_between_hubs(wide, cuda):
    """Two neighbours that share all others, by either way of adding."""
    import torch
    n = 100002
    leaves = np.arange(2, n)
    off = np.r_[0, n - 1, 2 * (n - 1), 2 * (n - 1) + 2 * np.arange(1, n - 1)].astype(np.int32)
    ind = np.concatenate([[1], leaves, [0], leaves, np.tile([0, 1], n - 2)]).astype(np.int32)
    w = ((1 + np.random.default_rng(4).integers(0, 1 << 24, n)) * 2.0 ** -24).astype(np.float32)
    if wide:
        w[7] = 2.0 ** -40
    g = api.DeviceCSR(n, torch.from_numpy(off).to(cuda), torch.from_numpy(ind).to(cuda))
    W = torch.from_numpy(w).to(cuda)
    assert api.weighted_sum_mode(g, W) == (api.SUM_DOUBLE_DOUBLE if wide else api.SUM_FP64)
    print(f"[gpu] two hubs wide={wide} n={n}", flush=True)
    out = api.jaccard(g, weights=W).cpu().numpy()
    x = w.astype(np.float64)
    common = x[2:].sum()
    assert abs(out[0] - common / x.sum()) <= 1e-6 and out[0] == out[n - 1]
    # (hub, leaf): the other hub is the one common neighbour
    ref = x[1] / ((common + x[1]) + (x[0] + x[1]) - x[1])
    assert np.all(np.abs(out[1:n - 1] - ref) <= 1e-6 * ref)
