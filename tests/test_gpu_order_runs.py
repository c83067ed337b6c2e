"""Short processing orders (runs of 1024 sites sorted by a workgroup each and merged by rank) against a stable sort by numpy, at the
edges of a wavefront's and a workgroup's run; inserts on both sides of what one workgroup ranks."""
import ctypes

import numpy as np
import pytest
import torch

from workloads import scenes

pytestmark = pytest.mark.gpu
I64 = ctypes.c_int64


def metadata(pts, capacity):
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    m = S.Metadata_3()
    m._bind(torch.device("cuda:0"))
    sc = m.scale((4096,) * 3, create_capacity=capacity)
    m.insert(sc, torch.from_numpy(np.ascontiguousarray(pts, np.int32)).cuda())
    return m, sc


def spread(v):
    return sum(((v >> b) & 1) << (3 * b) for b in range(4))


@pytest.mark.parametrize("n", [1, 64, 65, 1023, 1024, 1025, 2048, 2049, 7169, 8191])
@pytest.mark.parametrize("captured", [False, True])
def test_order_of_short_scales(n, captured):
    from sparseconvnet._lib import lib, ptr, stream_ptr

    n_old = 4500
    pts = scenes.boxes_scene(seed=n, n=n_old + n).astype(np.int32)
    pts[:, :3] += 61  # (several blocks of 64^3)
    m, sc = metadata(pts, n_old + n)
    assert sc.n == n_old + n
    m.ssc_rulebook((4096,) * 3)
    nbr = sc.nbr.t
    order = torch.full((sc.n,), -5, dtype=torch.int32, device="cuda")
    call = lambda: lib.insc_order_build(sc.grid, ptr(nbr), I64(n_old), I64(n), ptr(order), stream_ptr())
    if captured:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
        for _ in range(3):
            order.fill_(-5)
            graph.replay()
    else:
        call()
    c = sc.coords_view().cpu().numpy()[n_old:].astype(np.int64)
    has = nbr[n_old:sc.n].cpu().numpy() >= 0
    pattern = (has.astype(np.int64) << np.arange(27)).sum(1)
    mort = spread((c[:, 0] >> 6) & 15) | spread((c[:, 1] >> 6) & 15) << 1 | spread((c[:, 2] >> 6) & 15) << 2
    key = ((c[:, 3] & 1) << 39) | (mort << 27) | pattern
    got = order.cpu().numpy()
    assert (got[:n_old] == -5).all()
    assert (got[n_old:] == n_old + np.argsort(key, kind="stable")).all()


@pytest.mark.parametrize("P", [4095, 4096, 4097, 7168, 7169, 16384, 16385])
def test_inserts_around_what_one_workgroup_ranks(orc, P):
    rng = np.random.default_rng(P)
    pts = np.concatenate([rng.integers(0, 22, (2 * P, 3)), np.zeros((2 * P, 1), np.int64)], 1).astype(np.int32)  # many repeats
    m, sc = metadata(pts[:P], 2 * P)
    sop, osc, _ = orc.grid_build(pts[:P])
    assert (sc.coords_view().cpu().numpy() == osc).all()
    both = m.insert(sc, torch.from_numpy(pts[P:]).cuda())  # (onto a grid that holds sites)
    sop, osc, _ = orc.grid_build(pts)
    assert (sc.coords_view().cpu().numpy() == osc).all()
    assert (both.cpu().numpy() == sop[P:]).all()


@pytest.mark.parametrize("P", [4000, 5000, 16384, 30000])
@pytest.mark.parametrize("cleared", [False, True])
def test_captured_inserts_meet_the_sites_of_the_launch_before(orc, P, cleared):
    """An insert captured while the grid was empty: launched again, it finds its own sites (unless the graph clears them)."""
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import lib, ptr, stream_ptr

    rng = np.random.default_rng(P)
    side = int(P ** (1 / 3)) + 1
    pts = np.concatenate([rng.integers(0, side, (P, 3)), np.zeros((P, 1), np.int64)], 1).astype(np.int32)
    m, sc = metadata(pts[::-1], 2 * P)  # (scratch memory for P rows)
    want, osc, _ = orc.grid_build(pts)
    c = torch.from_numpy(pts).cuda()
    sop = torch.empty(P, dtype=torch.int32, device="cuda")
    n = I64(0)
    clear = lambda: lib.insc_grid_clear(sc.grid, stream_ptr())
    clear()
    lib.insc_grid_size(sc.grid, ctypes.byref(n), stream_ptr())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        if cleared:
            clear()
        lib.insc_grid_insert(sc.grid, ptr(c), I64(P), ptr(sop), None, stream_ptr())
    for _ in range(3):
        sop.fill_(-5)
        graph.replay()
        torch.cuda.synchronize()
        count = S._from_ptr(lib.insc_grid_count_ptr(sc.grid), (1,), torch.int32, torch.device("cuda:0"))
        coords = S._from_ptr(lib.insc_grid_coords(sc.grid), (len(osc), 4), torch.int32, torch.device("cuda:0"))
        assert int(count[0]) == len(osc)
        assert (sop.cpu().numpy() == want).all() and (coords.cpu().numpy() == osc).all()
