"""Coordinate rows of every width and layout, widened and checked in one launch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cuda", [False, True])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.int16, torch.float64, torch.float32])
def test_coordinate_rows(dtype, cuda):
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    rng = np.random.default_rng(3)
    base = torch.from_numpy(rng.integers(0, 30000, (1025, 6))).to(dtype)
    base = base.cuda() if cuda else base
    for rows in (base[:, :4], base[:, 1:4], base[:, :3].contiguous(), base.t()[:4].t(), base[:1, :3].expand(257, 3), base[:1, 2:6],
                 base[:0, :3], base[::2, :3]):
        bad = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        got = S._coords4(rows, torch.device("cuda:0"), bad)
        torch.cuda.synchronize()
        want = torch.zeros((rows.shape[0], 4), dtype=torch.int32)
        want[:, :rows.shape[1]] = rows.cpu().to(torch.int32)
        assert got.is_contiguous() and torch.equal(got.cpu(), want) and int(bad[0]) == 0


# values whose low 32 bits are a coordinate among them
@pytest.mark.parametrize("cuda", [False, True])
@pytest.mark.parametrize("at,value,ok", [(0, -1, False), (1, 65535, True), (2, 65536, False), (3, 32767, True), (3, 32768, False),
                                         (3, -1, False), (0, 1 << 32, False), (0, (1 << 32) - 1, False), (1, -(1 << 40), False),
                                         (2, (1 << 32) + 9, False), (3, 7 - (1 << 33), False), (0, -(1 << 31), False)])
def test_coordinates_out_of_range(at, value, ok, cuda):
    from sparseconvnet import SCN as S

    rows = torch.zeros((700, 4), dtype=torch.int64)
    rows[699, at] = value
    bad = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    got = S._coords4(rows.cuda() if cuda else rows, torch.device("cuda:0"), bad)
    torch.cuda.synchronize()
    assert int(bad[0]) == (0 if ok else 1)
    assert bool((got[:699] == 0).all()) and (not ok or int(got[699, at]) == value)


@pytest.mark.parametrize("cuda", [False, True])
@pytest.mark.parametrize("value", [1 << 32, 5 - (1 << 33)])
def test_a_coordinate_beyond_32_bits_is_no_other_voxel(cuda, value):
    import sparseconvnet as scn
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import InscError
    from workloads.netdefs import NaiveUNet

    pts = torch.tensor([[0, 0, 0], [5, 0, 0], [7, 8, 9]])
    far = pts.clone()
    far[2, 0] = value
    pts, far = (pts.cuda(), far.cuda()) if cuda else (pts, far)
    t = S.Result_3()
    t.set(pts, torch.eye(3)[[2, 2, 2]])
    t.set(far[2:], torch.eye(3)[:1])
    with pytest.raises(InscError) as e:  # (by the next call that waits)
        len(t)
    assert e.value.code == -5
    assert t.multiQuery(far[2:]).item() == t.multiQuery(far[2:] * 0 + 999).item()  # (no such voxel)
    assert t.multiQuery(pts).tolist() == [2, 2, 2]
    feats = torch.ones((3, 3), device="cuda")
    layer = scn.InputLayer(3, 4096, mode=4)
    with pytest.raises(InscError) as e:
        layer([far, feats, 1])
    assert e.value.code == -5
    net = scn.compile(NaiveUNet(m=16, levels=2, seed=1).cuda().sparseModel, capacity_sites=4096)
    with torch.no_grad():
        net([pts, feats, 1], increment=False)
        with pytest.raises(InscError) as e:
            net([far, feats, 1], increment=True)
    assert e.value.code == -5


# frames ranked by one workgroup a scale and, beyond 16384 points, by the passes over the chip
@pytest.mark.parametrize("n,cols", [(300, 3), (2000, 4), (17000, 3), (17000, 4)])
def test_a_frame_reads_coordinates_of_any_type(n, cols):
    import sparseconvnet as scn
    from workloads.netdefs import NaiveUNet

    g = torch.Generator().manual_seed(n + cols)
    rows = torch.cat([torch.randint(0, 2 * int(n ** (1 / 3)), (n, 3), generator=g) + torch.tensor([0, 65000, 300]),
                      torch.randint(0, 3, (n, 1), generator=g)], 1)[:, :cols]
    feats = torch.rand((n, 3), generator=g).cuda()
    net = scn.compile(NaiveUNet(m=16, levels=3, seed=1).cuda().sparseModel, capacity_sites=2 * n, residual=True)
    forms = [lambda t: t.cuda().to(torch.int32), lambda t: t, lambda t: t.cuda(), lambda t: t.cuda().float(), lambda t: t.float(),
             lambda t: t.repeat(1, 2)[:, :cols], lambda t: t.to(torch.int32)]
    k = n // 3
    outs = []
    with torch.no_grad():
        for form in forms:
            outs.append([net([form(rows[:n - k]), feats[:n - k], 3], increment=False).clone(),
                         net([form(rows[n - 2 * k:]), feats[n - 2 * k:], 3], increment="residual").clone(),
                         net([form(rows[n - k:]), feats[n - k:], 3], increment=True, all_points=True).clone()])
    assert all(torch.equal(a, b) for o in outs[1:] for a, b in zip(outs[0], o))


def test_more_rows_than_threads_in_a_launch():
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init, lib, ptr, stream_ptr

    ensure_init(0)
    P = (1 << 28) + 257
    rows = torch.zeros((P, 3), dtype=torch.int32, device="cuda")
    rows[-1] = torch.tensor([4, 5, 6])
    rows[1 << 28, 1] = -3
    out = torch.full((P, 4), -9, dtype=torch.int32, device="cuda")
    bad = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    lib.insc_coords4(ptr(rows), 32, 3, S.I64(3), S.I64(P), ptr(out), ptr(bad), stream_ptr())
    torch.cuda.synchronize()
    assert int(bad[0]) == 1
    assert out[-1].tolist() == [4, 5, 6, 0] and out[1 << 28].tolist() == [0, -3, 0, 0]
    assert all(torch.equal(a[:, :3], b) and not bool(a[:, 3].any()) for a, b in zip(out.split(1 << 26), rows.split(1 << 26)))
