"""3^3 layers: whatever a launch's size makes of a tile - a wavefront for every partial sum, one for all of them, several
output blocks a wavefront, the kernels that share weights - a row's sum is formed the same way, bit for bit.  The packed
fp32 weights of the C ABI always run with one output block and, in narrow layers, one wavefront per tile: they are what the
others are compared with, and the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from workloads import scenes

pytestmark = pytest.mark.gpu
I64 = ctypes.c_int64
SZ = torch.LongTensor([4096, 4096, 4096])


def sites(C, n, seed):
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    pts = scenes.boxes_scene(seed=seed, n=n)
    m = S.Metadata_3()
    out = torch.empty(0, device="cuda")
    f = torch.from_numpy(np.random.default_rng(seed).normal(size=(len(pts), C)).astype(np.float32)).cuda()
    S.InputLayer_updateOutput(m, SZ, torch.from_numpy(pts.astype(np.int64)), f, out, 0, 4)
    return m, m.ssc_rulebook(SZ), pts, out


def run(m, sc, x, W, Cout, bias, raw=True, plan=True, rows=None):
    from sparseconvnet._lib import lib, ptr, stream_ptr

    Cin = x.shape[1]
    wp = None
    if not raw:
        wp = torch.empty(lib.insc_conv_packed_floats(27, Cin, Cout), device="cuda")
        lib.insc_conv_pack_weights(ptr(W), 27, Cin, Cout, ptr(wp), stream_ptr())
    out = torch.full((x.shape[0], Cout + 3), 7.0, device="cuda")[:, :Cout]  # (a row stride of its own)
    w = (ptr(W) if raw else None, None if raw else ptr(wp))
    if plan:
        p = m.ssc_plan(sc)
        lib.insc_conv_ssc_plan(ptr(x), I64(Cin), I64(sc.n), ptr(out), I64(Cout + 3), w[0], w[1], ptr(bias), ptr(sc.nbr.t), ptr(p[0]),
                               I64(p[2]), ptr(p[1]), ptr(p[3]), ptr(sc.order.t), None, I64(sc.n), Cin, Cout, stream_ptr())
    else:
        n = sc.n if rows is None else rows.numel()
        lib.insc_conv_nbr(ptr(x), I64(Cin), I64(sc.n), ptr(out), I64(Cout + 3), w[0], w[1], ptr(bias), ptr(sc.nbr.t), 27,
                          None if rows is None else ptr(rows), None, I64(n), Cin, Cout, None, stream_ptr())
    return out


# one chunk and two, a half chunk, one to three output blocks, a ragged one; the last five: too many tiles for a wavefront per sum
@pytest.mark.parametrize("Cin,Cout,n", [(16, 16, 700), (32, 32, 5000), (32, 20, 33), (48, 48, 3000), (48, 100, 1900), (16, 72, 31),
                                        (48, 48, 70000), (16, 96, 45000), (48, 90, 45000), (48, 100, 34000), (32, 130, 28000)])
def test_narrow_layers(orc, Cin, Cout, n):
    from sparseconvnet._lib import lib

    m, sc, pts, x = sites(Cin, n, seed=Cin + Cout)
    g = torch.Generator(device="cuda").manual_seed(n)
    W = torch.randn((27, Cin, Cout), generator=g, device="cuda") * (2.0 / Cin / 27) ** 0.5
    b = torch.randn(Cout, generator=g, device="cuda")
    got = run(m, sc, x, W, Cout, b)
    try:
        lib.insc_conv_set_filter_lds_min_tiles(1 << 40)  # one wavefront per tile
        want = run(m, sc, x, W, Cout, b, raw=False)
        assert torch.equal(got, want)
        assert torch.equal(run(m, sc, x, W, Cout, b, plan=False), want)
        lib.insc_conv_set_filter_lds_min_tiles(1)  # the filter in LDS, where there is such a kernel
        for raw in (True, False):
            assert torch.equal(run(m, sc, x, W, Cout, b, raw=raw), want)
    finally:
        lib.insc_conv_reset_launch_policy()
    rows = torch.randperm(sc.n, generator=g, device="cuda")[:max(1, min(sc.n // 2, 1000))].to(torch.int32)
    some = run(m, sc, x, W, Cout, b, plan=False, rows=rows)
    assert torch.equal(some[rows.long()], want[rows.long()])
    if n <= 5000:
        _, osc, _ = orc.grid_build(pts)
        _, counts, pairs = orc.ssc_rules(osc)
        ref, _ = orc.conv_forward(x.cpu().numpy(), W.cpu().numpy(), b.cpu().numpy(), pairs, counts, len(osc))
        np.testing.assert_allclose(got.cpu().numpy(), ref, rtol=1e-4, atol=1e-5)


# two output blocks a wavefront, three, over one and several blocks of wavefronts; widths that end inside a block
@pytest.mark.parametrize("Cin,Cout,n", [(64, 64, 20000), (80, 96, 20000), (96, 90, 20000), (112, 100, 20000), (128, 128, 6000),
                                        (192, 96, 10500), (160, 128, 4000)])
def test_several_output_blocks_a_wavefront(Cin, Cout, n):
    from sparseconvnet._lib import lib

    m, sc, _, x = sites(Cin, n, seed=Cin + Cout)
    g = torch.Generator(device="cuda").manual_seed(n)
    W = torch.randn((27, Cin, Cout), generator=g, device="cuda") * (2.0 / Cin / 27) ** 0.5
    b = torch.randn(Cout, generator=g, device="cuda")
    try:
        lib.insc_conv_set_shared_weights_min_units(1 << 40)
        lib.insc_conv_set_wavefront_per_unit_min_units(1 << 40)
        want = run(m, sc, x, W, Cout, b, raw=False)
        assert torch.equal(run(m, sc, x, W, Cout, b), want)
        assert torch.equal(run(m, sc, x, W, Cout, b, plan=False), want)
        x[7, Cin - 1] = float("inf")  # (sums that are formed again, in every block of columns)
        assert torch.equal(run(m, sc, x, W, Cout, b).nan_to_num(3.0), run(m, sc, x, W, Cout, b, raw=False).nan_to_num(3.0))
    finally:
        lib.insc_conv_reset_launch_policy()
    rows = torch.randperm(sc.n, generator=g, device="cuda")[:500].to(torch.int32)  # (too few tiles for it)
    x[7, Cin - 1] = 0.5
    full = run(m, sc, x, W, Cout, b)
    assert torch.equal(run(m, sc, x, W, Cout, b, plan=False, rows=rows)[rows.long()], full[rows.long()])
