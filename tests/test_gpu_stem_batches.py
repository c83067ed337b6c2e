"""3^3 layers of one to four input channels: batches of rows are fetched one by one or ahead of the one that is computed.  Row
counts around a batch, widths that take one and two (row, offset) pairs a thread, row lists and an absent neighbour next to
weights that are not finite, against 64-bit sums; and both forms against each other, where a block has many batches."""
import numpy as np
import pytest
import torch

from workloads import scenes

pytestmark = pytest.mark.gpu
SZ = torch.LongTensor([4096, 4096, 4096])


@pytest.fixture(scope="module")
def scene():
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    pts = scenes.boxes_scene(seed=11, n=20000)
    m = S.Metadata_3()
    out = torch.empty(0, device="cuda")
    S.InputLayer_updateOutput(m, SZ, torch.from_numpy(pts.astype(np.int64)), torch.ones((len(pts), 1), device="cuda"), out, 0, 4)
    sc = m.ssc_rulebook(SZ)
    return m, sc.nbr.t[:sc.n].contiguous()


@pytest.mark.parametrize("cin,cout", [(1, 16), (2, 256), (3, 32), (3, 20), (3, 100), (4, 16), (4, 48)])
@pytest.mark.parametrize("n_rows", [1, 7, 8, 9, 33, 9000, None])
def test_stem(scene, cin, cout, n_rows):
    from sparseconvnet.SCN import I64, lib, ptr, stream_ptr

    _, nbr = scene
    n = len(nbr)
    rng = np.random.default_rng(cin * 1000 + cout)
    x, W, b = (rng.standard_normal(s).astype(np.float32) for s in ((n, cin), (27, cin, cout), (cout,)))
    rows = rng.permutation(n)[:n_rows].astype(np.int32)
    W[5, 0, 0] = np.inf  # reaches only rows that have the offset
    xd, Wd, bd, rd = (torch.from_numpy(a).cuda() for a in (x, W, b, rows))
    out = torch.full((n, cout), 7.0, device="cuda")
    lib.insc_conv_nbr(ptr(xd), I64(cin), I64(n), ptr(out), I64(cout), ptr(Wd), None, ptr(bd), ptr(nbr), 27, ptr(rd), None,
                      I64(len(rows)), cin, cout, None, stream_ptr())
    got, ids = out.cpu().numpy(), nbr.cpu().numpy()
    untouched = np.setdiff1d(np.arange(n), rows)
    assert (got[untouched] == 7.0).all()
    ref, size = np.tile(b.astype(np.float64), (n, 1)), np.tile(np.abs(b).astype(np.float64), (n, 1))
    for k in range(27):
        i = np.flatnonzero(ids[:, k] >= 0)
        ref[i] += x[ids[i, k]].astype(np.float64) @ W[k].astype(np.float64)
        size[i] += np.abs(x[ids[i, k]]).astype(np.float64) @ np.abs(W[k]).astype(np.float64)
    ref, got, size = ref[rows], got[rows], size[rows]
    fin = np.isfinite(ref)
    assert (fin[:, 1:]).all() and not fin[:, 0].all() or len(rows) < 100
    assert (got[~fin] == ref[~fin]).all()
    # (one rounding per product-and-add: at most 27 * cin + 1 of half a unit each of a sum no larger than `size`)
    assert (np.abs(got - ref)[fin] <= (27 * cin + 1) * 2.0 ** -24 * size[fin]).all()


# each form that runs ahead of its batch: 256 / cout rows a batch (16 at most), 2048 blocks, five or twelve batches each and a bit
@pytest.mark.parametrize("cin,cout,n", [(1, 256, 24581), (2, 16, 163845), (2, 20, 122885), (2, 128, 20487), (3, 90, 4100),
                                        (4, 64, 40970)])
def test_a_batch_ahead_gives_the_same_bits(cin, cout, n):
    from sparseconvnet.SCN import I64, lib, ptr, stream_ptr

    g = torch.Generator(device="cuda").manual_seed(n)
    nbr = torch.randint(-2 * n, n, (n, 27), generator=g, device="cuda", dtype=torch.int32).clamp_(min=-1)
    x = torch.randn((n, cin), generator=g, device="cuda")
    W = torch.randn((27, cin, cout), generator=g, device="cuda")
    b = torch.randn(cout, generator=g, device="cuda")
    order = torch.randperm(n, generator=g, device="cuda").to(torch.int32)

    def run(rows):
        out = torch.full((n, cout), 7.0, device="cuda")
        for r in rows:
            lib.insc_conv_nbr(ptr(x), I64(cin), I64(n), ptr(out), I64(cout), ptr(W), None, ptr(b), ptr(nbr), 27, ptr(r), None,
                              I64(len(r)), cin, cout, None, stream_ptr())
        return out

    many, few = run([order]), run(order.split(1000))
    ref, size = b.double().repeat(n, 1), b.double().abs().repeat(n, 1)
    for k in range(27):
        at = (nbr[:, k] >= 0).nonzero()[:, 0]
        xk = x[nbr[at, k].long()].double()
        ref[at] += xk @ W[k].double()
        size[at] += xk.abs() @ W[k].double().abs()
    for got in (many, few):
        assert bool(((got.double() - ref).abs() <= (27 * cin + 1) * 2.0 ** -24 * size).all())
    assert torch.equal(many, few)
