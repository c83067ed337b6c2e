"""Processing orders of scales on both sides of the sizes where the shared radix passes change (blocks of 2048 pairs, 256
blocks at most): the whole network on the shared launches must give the bits of the module tree, whose scales are
sorted one by one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [262144, 262145, 300001, 524288])
def test_shared_radix_passes_beyond_128_blocks(n):
    import sparseconvnet as scn
    from workloads.netdefs import NaiveUNet

    side = 1
    while side * side < n:
        side += 1
    pts = np.stack([np.arange(n) // side, np.arange(n) % side, np.zeros(n, np.int64)], 1) + 512  # n distinct sites exactly
    pts[:, 2] += (pts[:, 0] // 7) % 3
    pts = pts[np.random.default_rng(n).permutation(n)]
    x = [torch.from_numpy(pts), torch.from_numpy(np.random.default_rng(1).random((n, 3), np.float32)).cuda(), 1]
    model = NaiveUNet(m=16, levels=2, seed=3).cuda()
    with torch.no_grad():
        got = scn.compile(model.sparseModel, capacity_sites=600000)(x, increment=False).clone()
        prev = scn.set_auto_compile(False)
        try:
            want = model.sparseModel(x)
        finally:
            scn.set_auto_compile(prev)
    assert got.shape[0] == n and torch.equal(got, want)
