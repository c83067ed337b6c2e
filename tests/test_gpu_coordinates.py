"""Coordinate rows of every width and layout, widened and checked in one launch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cuda", [False, True])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.int16, torch.float64])
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


@pytest.mark.parametrize("at,value,ok", [(0, -1, False), (1, 65535, True), (2, 65536, False), (3, 32767, True), (3, 32768, False),
                                         (3, -1, False), (0, 1 << 32, True), (0, (1 << 32) - 1, False)])
def test_coordinates_out_of_range(at, value, ok):
    from sparseconvnet import SCN as S

    rows = torch.zeros((700, 4), dtype=torch.int64)
    rows[699, at] = value  # (narrowed to 32 bits first, as ever)
    bad = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    S._coords4(rows, torch.device("cuda:0"), bad)
    torch.cuda.synchronize()
    assert int(bad[0]) == (0 if ok else 1)
