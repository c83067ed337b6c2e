"""A destroyed grid's memory serves the grids made after it: nothing of the old scene may show, whatever the sizes,
streams and threads involved."""
import threading

import numpy as np
import pytest
import torch

from workloads import scenes

pytestmark = pytest.mark.gpu
SZ = torch.LongTensor([4096, 4096, 4096])


def structure(pts):
    """Site ids, coordinates and 3^3 map of a scene, on the current stream; the grid is dropped afterwards."""
    from sparseconvnet import SCN as S

    m = S.Metadata_3()
    out = torch.empty(0, device="cuda")
    S.InputLayer_updateOutput(m, SZ, torch.from_numpy(pts.astype(np.int64)), torch.ones((len(pts), 1), device="cuda"), out, 0, 4)
    sc = m.ssc_rulebook(SZ)
    return sc.coords_view().cpu().numpy().copy(), sc.nbr.t[:sc.n].cpu().numpy().copy()


def expect(orc, pts):
    _, sc, _ = orc.grid_build(pts)
    return sc


@pytest.mark.parametrize("sizes", [(3000, 3000, 2900, 3100), (40000, 500, 40000, 41000), (1, 60000, 1, 3000)])
def test_a_new_grid_holds_nothing_of_an_old_one(orc, sizes):
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    for i, n in enumerate(sizes):
        pts = scenes.boxes_scene(seed=20 + i, n=n)
        coords, nbr = structure(pts)
        sc = expect(orc, pts)
        assert (coords == sc).all()
        index = {tuple(c): j for j, c in enumerate(sc.tolist())}
        for row in np.random.default_rng(i).integers(0, len(sc), 50):
            x, y, z, b = sc[row].tolist()
            want = [index.get((x + a, y + c, z + d, b), -1) for a in (-1, 0, 1) for c in (-1, 0, 1) for d in (-1, 0, 1)]
            assert nbr[row].tolist() == want


def test_threads_and_streams_share_the_pool(orc):
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    clouds = [scenes.boxes_scene(seed=40 + i, n=4000 + 300 * i) for i in range(3)]
    want = [expect(orc, p) for p in clouds]
    bad = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(4):
                    coords, _ = structure(clouds[i])
                    if not (coords == want[i]).all():
                        bad.append(i)
        except Exception as e:  # (an assertion in a thread would go unseen)
            bad.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def _busy(ms=40):
    """Work of about that many milliseconds queued on the current stream."""
    a = torch.randn(4096, 4096, device="cuda")
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    a @ a
    torch.cuda.synchronize()
    e[0].record()
    a @ a
    e[1].record()
    torch.cuda.synchronize()
    n = int(ms / e[0].elapsed_time(e[1])) + 1
    for _ in range(n):
        a @ a


def test_creation_does_not_wait_for_queued_work():
    import ctypes
    import time

    from sparseconvnet._lib import ensure_init, lib

    ensure_init(0)
    for _ in range(2):  # (the first grid of a size may have to allocate)
        g = ctypes.c_void_p()
        _busy()
        t0 = time.perf_counter()
        lib.insc_grid_create(ctypes.c_int64(200000), ctypes.byref(g))
        t1 = time.perf_counter()
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        lib.insc_grid_destroy(g)
    assert t1 - t0 < 0.25 * (t2 - t0), "creation took %.1f of %.1f ms" % ((t1 - t0) * 1e3, (t2 - t0) * 1e3)


@pytest.mark.parametrize("n", [3000, 60000])
def test_a_new_grid_is_cleared_before_any_stream_uses_it(orc, n):
    """Work is queued on the null stream, where a new grid's clearing waits behind it; another stream inserts into the grid
    and queries it meanwhile."""
    import ctypes

    from sparseconvnet._lib import ensure_init, lib, ptr, stream_ptr

    ensure_init(0)
    I64 = ctypes.c_int64
    side = torch.cuda.Stream()
    for seed in range(3):  # (the second and third grid take the first one's memory)
        pts = scenes.boxes_scene(seed=70 + seed, n=n)
        sop, sc, _ = orc.grid_build(pts)
        c4 = np.zeros((n, 4), np.int32)
        c4[:, :pts.shape[1]] = pts
        d = torch.from_numpy(c4).cuda()
        site = torch.empty(n, dtype=torch.int32, device="cuda")
        found = torch.empty(n, dtype=torch.int32, device="cuda")
        empty = torch.empty(n, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        _busy(20)
        a, b, count = ctypes.c_void_p(), ctypes.c_void_p(), I64(0)
        lib.insc_grid_create(I64(n), ctypes.byref(a))
        lib.insc_grid_create(I64(n), ctypes.byref(b))
        with torch.cuda.stream(side):
            lib.insc_grid_query(b, ptr(d), I64(n), ptr(empty), stream_ptr())
            lib.insc_grid_insert(a, ptr(d), I64(n), ptr(site), ctypes.byref(count), stream_ptr())
            lib.insc_grid_query(a, ptr(d), I64(n), ptr(found), stream_ptr())
        torch.cuda.synchronize()
        assert count.value == len(sc) and (site.cpu().numpy() == sop).all() and (found.cpu().numpy() == sop).all()
        assert (empty.cpu().numpy() == -1).all()
        lib.insc_grid_destroy(a)
        lib.insc_grid_destroy(b)


def test_the_kept_memory_is_given_back():
    import sparseconvnet as scn
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    scn.empty_cache()
    torch.cuda.synchronize()
    structure(scenes.boxes_scene(seed=3, n=60000))
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    structure(scenes.boxes_scene(seed=3, n=60000))
    torch.cuda.empty_cache()
    assert torch.cuda.mem_get_info()[0] >= free  # (the second scene's grids took the first one's memory)
    scn.empty_cache()
    assert torch.cuda.mem_get_info()[0] > free


def test_a_view_of_the_coordinates_keeps_its_scene():
    """The memory of a scene whose coordinates are still looked at does not go to the next scene."""
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)

    def scene(seed):
        pts = scenes.boxes_scene(seed=seed, n=5000)
        m = S.Metadata_3()
        out = torch.empty(0, device="cuda")
        S.InputLayer_updateOutput(m, SZ, torch.from_numpy(pts.astype(np.int64)), torch.ones((len(pts), 1), device="cuda"), out, 0, 4)
        return m

    m = scene(90)
    view = m.scale(SZ).coords_view()
    want = view.cpu().numpy().copy()
    del m
    others = [scene(91 + i) for i in range(3)]
    assert (view.cpu().numpy() == want).all()
    assert not (others[0].scale(SZ).coords_view()[:100].cpu().numpy() == want[:100]).all()
    m = scene(95)
    part = m.scale(SZ).coords_view()[7:9]  # (a slice of a view is one as well)
    want = part.cpu().numpy().copy()
    m.clear()
    others += [scene(96), scene(97)]
    assert (part.cpu().numpy() == want).all()


def test_growing_grids_take_and_leave_kept_memory(orc):
    """A grid that is inserted into piece by piece outgrows its table, coordinates and scratch memory several times; a second
    one takes over what the first outgrew and needs no more of the device."""
    import ctypes

    import sparseconvnet as scn
    from sparseconvnet._lib import ensure_init, lib, ptr, stream_ptr

    ensure_init(0)
    scn.empty_cache()
    I64 = ctypes.c_int64
    pts = scenes.boxes_scene(seed=33, n=60000)
    sop, sc, _ = orc.grid_build(pts)
    c4 = np.zeros((len(pts), 4), np.int32)
    c4[:, :pts.shape[1]] = pts
    d = torch.from_numpy(c4).cuda()
    site = torch.empty(len(pts), dtype=torch.int32, device="cuda")
    free = []
    for _ in range(3):
        g, n = ctypes.c_void_p(), I64(0)
        lib.insc_grid_create(I64(1024), ctypes.byref(g))
        a = 0
        for step in (500, 3000, 9000, 20000, len(pts)):
            b = min(a + step, len(pts))
            lib.insc_grid_insert(g, ptr(d[a:b]), I64(b - a), ptr(site[a:b]), ctypes.byref(n), stream_ptr())
            a = b
        assert n.value == len(sc) and (site.cpu().numpy() == sop).all()
        lib.insc_grid_query(g, ptr(d), I64(len(pts)), ptr(site), stream_ptr())
        assert (site.cpu().numpy() == sop).all()
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
        lib.insc_grid_destroy(g)
    assert free[1] == free[2]
