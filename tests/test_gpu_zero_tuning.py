"""A tuning of zeros is no tuning: the same way to the result as a call without
one, at every size where that way changes."""
import numpy as np
import pytest

from jaccard_amd import api, graphs

pytestmark = pytest.mark.gpu

GRAPHS = {"lds": lambda: graphs.rmat(9, 8, seed=2), "owner": lambda: graphs.rmat(13, 16, seed=2),
          "oriented": lambda: graphs.rmat(18, 24, seed=2)}


def kernels(dg, W, tuning):
    api.profile_reset()
    api.profile_enable(True)
    out = api.jaccard(dg, weights=W, tuning=tuning)
    api.profile_enable(False)
    used = {k for k in api.profile_names() if api.profile_query(k)[0] > 0}
    api.profile_reset()
    return out, used


@pytest.mark.parametrize("name", list(GRAPHS))
def test_zeros_are_the_default(name, cuda):
    import torch
    g = GRAPHS[name]()
    dg = api.DeviceCSR.from_host(g, cuda)
    w = ((1 + np.random.default_rng(3).integers(0, 1 << 24, g.n)) * 2.0 ** -24).astype(np.float32)
    for W in (None, torch.from_numpy(w).to(cuda)):
        print(f"[gpu] zero tuning {name} n={g.n} m={g.m}", flush=True)
        want, default = kernels(dg, W, None)
        out, used = kernels(dg, W, {})
        assert used == default and ("tiny" in used) == (name == "lds") and ("tri_wedge" in used) == (name == "oriented")
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
        # a field of the owner engine's names that engine
        out, used = kernels(dg, W, dict(small_blocks_per_cu=16))
        assert "owner_small" in used and "tiny" not in used and "tri_wedge" not in used
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
