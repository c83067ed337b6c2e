"""fp32 products as sums of bf16 products (csrc/conv.hip): what such a sum can get wrong - infinities and NaN,
magnitudes far from one, the error against 64-bit sums - on every matrix-core kernel."""
import numpy as np
import pytest
import torch

from workloads import scenes

pytestmark = pytest.mark.gpu
SZ = torch.LongTensor([4096, 4096, 4096])
NEVER = 1 << 40
# (Cin, Cout, filter-in-LDS from, wavefront per unit from, shared weights from): one kernel each
KERNELS = [(16, 16, 1, NEVER, NEVER), (32, 32, 1, NEVER, NEVER), (32, 20, NEVER, NEVER, NEVER), (48, 64, NEVER, NEVER, NEVER),
           (64, 64, NEVER, 1, NEVER), (64, 96, NEVER, NEVER, 1), (80, 32, NEVER, NEVER, 1), (96, 64, NEVER, NEVER, NEVER),
           (128, 128, NEVER, NEVER, NEVER), (160, 100, NEVER, NEVER, NEVER)]


@pytest.fixture(scope="module")
def scene():
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    pts = scenes.boxes_scene(seed=7, n=2300)
    m = S.Metadata_3()
    out = torch.empty(0, device="cuda")
    S.InputLayer_updateOutput(m, SZ, torch.from_numpy(pts.astype(np.int64)), torch.ones((len(pts), 1), device="cuda"), out, 0, 4)
    sc = m.ssc_rulebook(SZ)
    return S, m, sc, sc.nbr.t[:sc.n].cpu().numpy()


def layer(scene, x, W, b, case, n_in=None, events=None):
    from sparseconvnet._lib import lib

    S, m, sc, _ = scene
    out = torch.full((sc.n, W.shape[2]), 7.0, device="cuda")
    xd, Wd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(), torch.from_numpy(b).cuda()
    plan = m.ssc_plan(sc)
    try:
        lib.insc_conv_set_filter_lds_min_tiles(case[2])
        lib.insc_conv_set_wavefront_per_unit_min_units(case[3])
        lib.insc_conv_set_shared_weights_min_units(case[4])
        S.packed_weight(Wd, 27)
        if events is not None:
            events += [torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)]
            torch.cuda.synchronize()
            events[0].record()
        S.ssc_rows_planned(xd[:n_in], out, Wd, bd, sc, plan)
        if events is not None:
            events[1].record()
    finally:
        lib.insc_conv_reset_launch_policy()
    return out.cpu().numpy()


def sums64(nbr, x, W, b):
    ref = np.tile(b.astype(np.float64), (len(nbr), 1))
    for k in range(27):
        i = np.flatnonzero(nbr[:, k] >= 0)
        with np.errstate(invalid="ignore"):
            ref[i] += x[nbr[i, k]].astype(np.float64) @ W[k].astype(np.float64)
    return ref


def data(scene, case):
    rng = np.random.default_rng(case[0] + case[1])
    n = scene[2].n
    x = rng.normal(size=(n, case[0])).astype(np.float32)
    W = (rng.normal(size=(27,) + case[:2]) * (2.0 / case[0] / 27) ** 0.5).astype(np.float32)
    return rng, x, W, rng.normal(size=case[1]).astype(np.float32)


@pytest.mark.parametrize("case", KERNELS)
def test_error_against_64_bit_sums(scene, case):
    """Per element: each fp32 rounding of the running sum is half a unit in the last place of a partial sum, which
    |b| + sum |x||w| bounds; there are at most 27 * Cin / 8 of them in a fp32 chain of this length."""
    _, x, W, b = data(scene, case)
    got, nbr = layer(scene, x, W, b, case), scene[3]
    ref, mag = sums64(nbr, x, W, b), sums64(nbr, np.abs(x), np.abs(W), np.abs(b))
    err = np.abs(got - ref)
    assert (err <= 2.0 ** -24 * 27 * case[0] / 8 * mag).all()
    # and over all of them: no more than a chain of fp32 multiply-adds, which rounds its sum once per product, shows on
    # a sample of the same rows (here it is rounded once per 16 channels: a quarter of that is expected)
    some = np.random.default_rng(1).integers(0, len(x), 200)
    acc = np.tile(b, (len(some), 1))
    for k in range(27):
        src = nbr[some, k]
        for ci in range(case[0]):
            step = (x[src, ci].astype(np.float64)[:, None] * W[k, ci].astype(np.float64) + acc).astype(np.float32)
            acc = np.where(src[:, None] >= 0, step, acc)
    assert np.linalg.norm(err[some]) <= np.linalg.norm(acc - ref[some])


@pytest.mark.parametrize("case", KERNELS)
def test_magnitudes_far_from_one(scene, case):
    """Powers of two move through exactly."""
    _, x, W, b = data(scene, case)
    base = layer(scene, x, W, b, case)
    for e in (-60, 60):
        s = np.float32(2.0 ** e)
        assert (layer(scene, x * s, W, b * s, case) == base * s).all()


@pytest.mark.parametrize("case", KERNELS)
def test_infinities_and_nan(scene, case):
    """An infinity stays one (three parts of it would be infinity minus infinity), NaN stays NaN, and no
    other row changes."""
    rng, x, W, b = data(scene, case)
    base = layer(scene, x, W, b, case)
    n = len(x)
    x[rng.integers(0, n, 5), rng.integers(0, case[0], 5)] = np.inf
    x[rng.integers(0, n, 5), rng.integers(0, case[0], 5)] = -np.inf
    x[rng.integers(0, n, 3), rng.integers(0, case[0], 3)] = np.nan
    got, ref = layer(scene, x, W, b, case), sums64(scene[3], x, W, b)
    assert np.isinf(ref).any() and np.isnan(ref).any()
    fin = np.isfinite(ref)
    assert (got[fin] == base[fin]).all()
    assert (np.isnan(got) == np.isnan(ref)).all() and (got[np.isinf(ref)] == ref[np.isinf(ref)]).all()
    # the largest floats: their upper halves would round to infinity
    _, x, W, b = data(scene, case)
    x[7, 0] = np.float32(3.4e38)
    W[:, 0, :] = np.clip(W[:, 0, :], -0.01, 0.01)
    W[13, 1, 0] = np.float32(-3.4e38)
    x[:, 1] = 0
    got, ref = layer(scene, x, W, b, case), sums64(scene[3], x, W, b)
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= 1e-5 * np.abs(ref) + 1e-4 * np.abs(sums64(scene[3], np.minimum(np.abs(x), 9), np.minimum(np.abs(W), 9), b))).all()


@pytest.mark.parametrize("Cin,Cout", [(16, 16), (48, 224), (96, 33)])
def test_raw_packed_and_split_weights_give_the_same_bits(scene, Cin, Cout):
    from sparseconvnet._lib import lib, ptr, stream_ptr

    S, m, sc, _ = scene
    _, x, W, b = data(scene, (Cin, Cout))
    xd, Wd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(), torch.from_numpy(b).cuda()
    packed = torch.empty(lib.insc_conv_packed_floats(27, Cin, Cout), device="cuda")
    split = torch.empty(lib.insc_conv_split_floats(27, Cin, Cout), device="cuda")
    lib.insc_conv_pack_weights(ptr(Wd), 27, Cin, Cout, ptr(packed), stream_ptr())
    lib.insc_conv_split_weights(ptr(Wd), 27, Cin, Cout, ptr(split), stream_ptr())
    got = []
    for raw, wp in ((ptr(Wd), None), (None, ptr(packed)), (None, ptr(split) | 1)):
        out = torch.full((sc.n, Cout), 7.0, device="cuda")
        lib.insc_conv_nbr(ptr(xd), Cin, sc.n, ptr(out), Cout, raw, wp, ptr(bd), ptr(sc.nbr.t), 27, None, None, sc.n, Cin, Cout,
                          None, stream_ptr())
        got.append(out)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("case", KERNELS)
def test_repeated_sums_read_inside_the_input_matrix(scene, case):
    """Map entries beyond n_in_rows count as rows of zeros (the gather is bounds-checked against it), also in the sums
    that are formed a second time because they are not finite."""
    S, m, sc, nbr = scene
    rng, x, W, b = data(scene, case)
    half = sc.n // 2
    x[rng.integers(0, half, 40), 0] = np.nan
    x[rng.integers(0, half, 40), 0] = np.inf
    x[half:] = 1e30  # (allocated, but not part of the matrix that is handed over)
    got = layer(scene, x, W, b, case, n_in=half)
    x[half:] = 0
    ref = sums64(nbr, x, W, b)
    assert np.isnan(ref).any() and np.isinf(ref).any()
    assert (np.isnan(got) == np.isnan(ref)).all() and (got[np.isinf(ref)] == ref[np.isinf(ref)]).all()
    fin = np.isfinite(ref)
    assert (np.abs(got[fin] - ref[fin]) <= 1e-4).all()


@pytest.mark.parametrize("case", KERNELS)
def test_a_layer_of_nan_costs_a_few_times_a_finite_one(scene, case):
    """One NaN of a scan reaches every site of the coarse scales: a layer whose sums are all repeated may take a few times
    as long (some ten at these sizes, where a finite layer is one short launch), not hundreds of times."""
    _, x, W, b = data(scene, case)

    def best(x):
        ts = []
        for _ in range(5):
            e = []
            layer(scene, x, W, b, case, events=e)
            ts.append(e[0].elapsed_time(e[1]))
        return min(ts)

    assert best(np.full_like(x, np.nan)) < 25 * best(x)


@pytest.mark.parametrize("case", KERNELS)
def test_an_infinite_weight_reaches_only_rows_that_have_its_offset(scene, case):
    """A row without a neighbour takes no part in that offset, whatever its tile mates do: zero times infinity does not
    come in.  (Its sum may be formed the other way, so it is compared within the error of a fp32 sum, not bit for bit.)"""
    _, x, W, b = data(scene, case)
    mag = sums64(scene[3], np.abs(x), np.abs(W), np.abs(b))
    W[3, 5, 1], W[26, 7, 0] = np.inf, -np.inf
    got, ref = layer(scene, x, W, b, case), sums64(scene[3], x, W, b)
    fin = np.isfinite(ref)
    assert np.isinf(ref).any() and (got[~fin] == ref[~fin]).all()
    assert (np.abs(got[fin] - ref[fin]) <= 2.0 ** -24 * 27 * case[0] * mag[fin]).all()


def sums64_through(maps, x, W, b):
    """Like sums64, for any map [rows, K] and several sources."""
    ref = np.tile(b.astype(np.float64), (len(maps[0]), 1))
    for nbr, src in zip(maps, x):
        for k in range(W.shape[0]):
            i = np.flatnonzero(nbr[:, k] >= 0)
            with np.errstate(invalid="ignore"):
                ref[i] += src[nbr[i, k]].astype(np.float64) @ W[k].astype(np.float64)
    return ref


@pytest.mark.parametrize("kind,Cin,Cout", [("nin", 48, 96), ("nin", 192, 64), ("down", 16, 32), ("down", 48, 70), ("down", 64, 96),
                                           ("up", 32, 16), ("up", 64, 40), ("up", 128, 64), ("incre", 32, 32),
                                           ("incre", 64, 40), ("incre", 128, 128), ("incre_up", 32, 16), ("incre_up", 96, 64)])
def test_the_other_maps(kind, Cin, Cout):
    """1x1, 2^3 stride-2, deconvolutions and the two sources of a residual frame, with infinities and NaN in some rows: every
    kernel has a form of its own for each map."""
    from sparseconvnet import SCN as S
    from sparseconvnet._lib import ensure_init

    ensure_init(0)
    rng = np.random.default_rng(Cin + Cout)
    vox = scenes.boxes_scene(seed=11, n=2600)
    old, new = vox[:1700], np.concatenate([vox[rng.choice(1700, 500, replace=False)], vox[1700:]])
    half = SZ // 2

    def sites(pts):
        m, e = S.Metadata_3(), torch.empty(0, device="cuda")
        S.InputLayer_updateOutput(m, SZ, torch.from_numpy(pts.astype(np.int64)), torch.ones((len(pts), 1), device="cuda"), e, 0, 4)
        return m

    m = sites(new)
    fine, coarse, d = m.down_rulebook(SZ, half)
    cpu = lambda t, n: t[:n].cpu().numpy()
    parent, off = cpu(d.parent.t, fine.n), cpu(d.offset.t, fine.n)
    K = {"nin": 1, "incre": 27}.get(kind, 8)
    W = (rng.normal(size=(K, Cin, Cout)) * (2.0 / Cin / K) ** 0.5).astype(np.float32)
    b = rng.normal(size=Cout).astype(np.float32)
    n_in = coarse.n if kind.endswith("up") else fine.n

    def spoil(x):
        x[rng.integers(0, len(x), 6), rng.integers(0, Cin, 6)] = np.inf
        x[rng.integers(0, len(x), 6), rng.integers(0, Cin, 6)] = -np.inf
        x[rng.integers(0, len(x), 4), rng.integers(0, Cin, 4)] = np.nan
        return x

    up = np.where(np.arange(8) == off[:, None], parent[:, None], -1)
    x = rng.normal(size=(n_in, Cin)).astype(np.float32)
    sets, maps = [x], {"nin": np.arange(fine.n)[:, None], "down": cpu(d.child.t, coarse.n), "up": up, "incre_up": up}
    if kind.startswith("incre"):
        ma = sites(old)
        _, coarse_a, _ = ma.down_rulebook(SZ, half)
        sets.append(rng.normal(size=(coarse_a.n if kind == "incre_up" else 1700, Cin)).astype(np.float32))
    if kind == "incre":
        maps = [cpu(m.ssc_rulebook(SZ).nbr.t, fine.n), cpu(m.incre_ssc_map(SZ, ma), fine.n)]
    elif kind == "incre_up":
        pe_c, pe_f = m.pre_exist_map(half, ma).cpu().numpy(), m.pre_exist_map(SZ, ma).cpu().numpy()
        maps = [up, np.where((up >= 0) & (pe_f < 0)[:, None], pe_c[up], -1)]
    else:
        maps = [maps[kind]]

    def run(sets):
        xs, Wd, bd = [torch.from_numpy(v).cuda() for v in sets], torch.from_numpy(W).cuda(), torch.from_numpy(b).cuda()
        out = torch.full((len(maps[0]), Cout), 7.0, device="cuda")
        two, e = torch.LongTensor([2, 2, 2]), torch.empty(0, device="cuda")
        if kind == "nin":
            S.NetworkInNetwork_updateOutput(xs[0], e, Wd[0], bd)
            return e.cpu().numpy()
        if kind == "down":
            S.conv_rows(xs[0], out, Wd, bd, d.child.t, 8, None, None, coarse.n)
        elif kind == "up":
            S.deconv_rows(xs[0], out, Wd, bd, d.parent.t, d.offset.t, None, None, fine.n)
        elif kind == "incre":
            S.Incre_SubmanifoldConvolution_updateOutput(SZ, torch.LongTensor([3, 3, 3]), m, xs[0], e, Wd, bd, ma, xs[1])
            return e.cpu().numpy()
        else:
            S.Incre_Deconvolution_updateOutput(half, SZ, two, two, m, xs[0], e, Wd, bd, ma, xs[1])
            return e.cpu().numpy()
        return out.cpu().numpy()

    base, ref = run(sets), sums64_through(maps, sets, W, b)
    mag = sums64_through(maps, [np.abs(v) for v in sets], np.abs(W), np.abs(b))
    assert (np.abs(base - ref) <= 2.0 ** -24 * (K * Cin / 8 + 2) * mag).all()
    bad = [spoil(v.copy()) for v in sets]
    got, ref = run(bad), sums64_through(maps, bad, W, b)
    fin = np.isfinite(ref)
    assert np.isnan(ref).any() and np.isinf(ref).any() and (got[fin] == base[fin]).all()
    assert (np.isnan(got) == np.isnan(ref)).all() and (got[np.isinf(ref)] == ref[np.isinf(ref)]).all()


@pytest.mark.parametrize("case", KERNELS)
@pytest.mark.parametrize("ex,ew", [(0, 0), (-104, 60), (-112, 60), (-126, 100), (-140, 100), (90, -112), (90, -126), (90, -140)])
def test_a_single_product_is_rounded_as_in_fp32(scene, case, ex, ew):
    """One input channel and the centre's offset alone: the result is one product, whatever the size of its factors
    (subnormal ones among them).  Its error is that of a fp32 product, half a unit in the last place, and at most 2^-27 of the
    product on top: 2^-30 from the part product that is left out and seven roundings of a sum of 2^-6 of it."""
    rng, x, W, b = data(scene, case)
    n = len(x)
    one, j = np.zeros_like(x), rng.integers(0, case[0], n)
    one[np.arange(n), j] = (x[np.arange(n), j].astype(np.float64) * 2.0 ** ex).astype(np.float32)
    Wc = np.zeros_like(W)
    Wc[13] = (W[13].astype(np.float64) * 2.0 ** ew).astype(np.float32)
    got, ref = layer(scene, one, Wc, np.zeros_like(b), case), one.astype(np.float64) @ Wc[13].astype(np.float64)
    err, fp32 = np.abs(got - ref), np.abs(ref.astype(np.float32) - ref)
    assert (err <= np.abs(ref) * (2.0 ** -24 + 2.0 ** -27)).all()
    assert np.linalg.norm(err) <= 1.02 * np.linalg.norm(fp32)


@pytest.mark.parametrize("case", KERNELS)
@pytest.mark.parametrize("ex,ew", [(-112, 60), (-126, 100), (-140, 100), (90, -126), (-60, -60), (100, 10), (10, 110), (60, 60)])
def test_error_against_64_bit_sums_far_from_one(scene, case, ex, ew):
    """The bound of test_error_against_64_bit_sums at both ends of the range, where parts of eight bits would run out of
    exponents (and, from sums of 2^82 and weights of 2^104 up, where the sums are formed in plain fp32: a rounding per
    product pair)."""
    rng, x, W, b = data(scene, case)
    x, W = ((v.astype(np.float64) * 2.0 ** e).astype(np.float32) for v, e in ((x, ex), (W, ew)))
    b = (b.astype(np.float64) * 2.0 ** (ex + ew)).astype(np.float32)
    got, nbr = layer(scene, x, W, b, case), scene[3]
    ref, mag = sums64(nbr, x, W, b), sums64(nbr, np.abs(x), np.abs(W), np.abs(b))
    assert (np.abs(got - ref) <= 2.0 ** -24 * 27 * case[0] / (8 if ex + ew < 70 and ew < 100 else 2) * mag).all()
