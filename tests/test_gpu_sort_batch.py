"""Processing orders of scales on both sides of the sizes where the shared radix passes change (blocks of 2048 pairs, 256
blocks at most): the sorted pairs themselves against a stable sort of the library, and the whole network on the shared
launches, which must give the bits of the module tree, whose scales are sorted one by one (bits that do not depend on the
order, as long as it names every site once)."""
import ctypes

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


class SortJob(ctypes.Structure):
    """insc::SortJob (csrc/common.h)"""
    _fields_ = [(f, ctypes.c_void_p) for f in ("keys", "vals_in", "vals_out", "inv_out")] + [("n", ctypes.c_int64)]


@pytest.mark.parametrize("sizes", [(262144, 2048, 1), (262145, 2049), (524288, 131072, 40000, 9000, 2047, 300, 33, 1), (499999, 500000)])
@pytest.mark.parametrize("bits", [8, 40])
def test_the_shared_passes_sort(sizes, bits):
    """The internal function, which no entry point reaches beyond 262144 pairs but the executor."""
    from sparseconvnet import _lib

    _lib.ensure_init(0)
    fn = getattr(_lib.cdll(), "_ZN4insc25sort_pairs_u64_into_batchEPKNS_7SortJobEiiP12ihipStream_t")
    fn.argtypes, fn.restype = [ctypes.POINTER(SortJob), ctypes.c_int, ctypes.c_int, ctypes.c_void_p], ctypes.c_int
    rng = np.random.default_rng(sum(sizes))
    jobs, keep = (SortJob * len(sizes))(), []
    for i, n in enumerate(sizes):
        # (few distinct high bits, as the patterns of a scene have: long runs of equal keys, whose order must stay)
        keys = torch.from_numpy(rng.integers(0, 1 << (bits if i % 2 else bits // 2), n, dtype=np.int64)).cuda()
        vals = torch.from_numpy(rng.permutation(n).astype(np.int32)).cuda()
        out, inv = torch.full_like(vals, -1), torch.full_like(vals, -1)
        want = vals[torch.sort(keys, stable=True).indices]
        jobs[i] = SortJob(keys.data_ptr(), vals.data_ptr(), out.data_ptr(), inv.data_ptr(), n)
        keep.append((keys, vals, out, inv, want))
    assert fn(jobs, len(sizes), bits, _lib.stream_ptr()) == 0
    torch.cuda.synchronize()
    for n, (_, _, out, inv, want) in zip(sizes, keep):
        assert torch.equal(out, want)
        assert torch.equal(inv[out.long()], torch.arange(n, dtype=torch.int32, device="cuda"))
