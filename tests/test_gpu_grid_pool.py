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
