"""Size-2 convolutions and deconvolutions: rows that 32-bit offsets reach are stored without a branch per row, rows of a
wider matrix one by one.  Both forms give the same bits, write nothing beside their rows and columns, and agree with the
sums in 64 bits."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
I64 = ctypes.c_int64
WIDE = (1 << 22) + 8  # floats per row: 16 MiB, more than 24-bit row strides


# a tile less a row, one and a row; ragged columns; one to four output blocks a wavefront, a tile over several; columns beyond
# the 1024 between the offset of a row that does not exist and 4 GB
@pytest.mark.parametrize("up", [False, True])
@pytest.mark.parametrize("Cin,Cout,n", [(32, 16, 31), (16, 33, 33), (48, 64, 1), (64, 90, 32), (32, 128, 70), (96, 40, 45), (96, 100, 5000), (32, 1060, 45), (96, 1060, 45)])
def test_rows_of_any_stride(Cin, Cout, n, up):
    from sparseconvnet._lib import ensure_init, lib, ptr, stream_ptr

    ensure_init(0)
    g = torch.Generator(device="cuda").manual_seed(n + Cin + up)
    n_in = n + 5
    x = torch.randn((n_in, Cin), generator=g, device="cuda")
    W = torch.randn((8, Cin, Cout), generator=g, device="cuda") * (1.0 / Cin) ** 0.5
    b = torch.randn(Cout, generator=g, device="cuda")
    wp = torch.empty(lib.insc_conv_packed_floats(8, Cin, Cout), device="cuda")
    lib.insc_conv_pack_weights(ptr(W), 8, Cin, Cout, ptr(wp), stream_ptr())
    nbr = torch.randint(-n_in, n_in, (n, 8), generator=g, device="cuda", dtype=torch.int32).clamp_(min=-1)
    parent = torch.randint(0, n_in, (n,), generator=g, device="cuda", dtype=torch.int32)
    offset = torch.randint(0, 8, (n,), generator=g, device="cuda", dtype=torch.int32)
    rows = torch.randperm(n, generator=g, device="cuda").to(torch.int32)[: max(1, n - 1)]

    def run(ld):
        store = torch.full(((n - 1) * ld + Cout + 1,), 7.0, device="cuda")
        out = torch.as_strided(store, (n, Cout + 1), (ld, 1))
        if up:
            lib.insc_deconv_down2(ptr(x), I64(Cin), I64(n_in), ptr(out), I64(ld), ptr(W), ptr(wp), ptr(b), ptr(parent), ptr(offset),
                                  ptr(rows), None, I64(rows.numel()), Cin, Cout, stream_ptr())
        else:
            lib.insc_conv_nbr(ptr(x), I64(Cin), I64(n_in), ptr(out), I64(ld), ptr(W), ptr(wp), ptr(b), ptr(nbr), 8, ptr(rows), None,
                              I64(rows.numel()), Cin, Cout, None, stream_ptr())
        return out

    got = run(Cout + 1)
    if n <= 70:
        assert torch.equal(run(WIDE), got)
    xd, Wd = x.double(), W.double()
    want, size = b.double().repeat(n, 1), b.double().abs().repeat(n, 1)
    for k in range(8):
        src = torch.where(offset == k, parent, -1) if up else nbr[:, k]
        at = (src >= 0).nonzero()[:, 0]
        xk = xd[src[at].long()]
        want[at] += xk @ Wd[k]
        size[at] += xk.abs() @ Wd[k].abs()
    done = torch.zeros(n, dtype=torch.bool, device="cuda")
    done[rows.long()] = True
    # 8 * Cin + 1 terms added in 32 bits, the products exact to 2^-22 of their size: (terms / 2 + 4) * 2^-23 of the sizes' sum
    bound = (4 * Cin + 5) * 2.0 ** -23 * size + 1e-30
    assert bool(((got[:, :Cout].double() - want).abs() <= bound)[done].all())
    assert bool((got[:, Cout] == 7.0).all()) and bool((got[~done] == 7.0).all())


# a row that begins below the reach of 32-bit offsets and ends beyond it, in one and in four wavefronts a tile
@pytest.mark.parametrize("Cin", [16, 96])
def test_a_row_that_crosses_the_reach_of_32_bit_offsets(Cin):
    from sparseconvnet._lib import ensure_init, lib, ptr, stream_ptr

    ensure_init(0)
    Cout, ld, n = 40000, 40004, 26842
    edge = 26840
    assert edge * ld * 4 < 0xFFFE0000 and edge * ld * 4 + Cout * 4 > 0xFFFFF000
    g = torch.Generator(device="cuda").manual_seed(Cin)
    x = torch.randn((64, Cin), generator=g, device="cuda")
    W = torch.randn((8, Cin, Cout), generator=g, device="cuda") * (1.0 / Cin) ** 0.5
    nbr = torch.randint(0, 64, (n, 8), generator=g, device="cuda", dtype=torch.int32)
    out = torch.full((n, ld), 7.0, device="cuda")

    def run(rows):
        r = torch.tensor(rows, dtype=torch.int32, device="cuda")
        lib.insc_conv_nbr(ptr(x), I64(Cin), I64(64), ptr(out), I64(ld), ptr(W), None, None, ptr(nbr), 8, ptr(r), None,
                          I64(len(rows)), Cin, Cout, None, stream_ptr())

    run([edge, 3])
    for r in (edge, 3):
        want, size = (sum(f(x[nbr[r, k].long()].double()) @ f(W[k].double()) for k in range(8)) for f in (lambda t: t, torch.abs))
        assert bool(((out[r, :Cout].double() - want).abs() <= (4 * Cin + 5) * 2.0 ** -23 * size + 1e-30).all())
    assert bool((out[:, Cout:] == 7.0).all())
    out[[edge, 3]] = 7.0
    assert bool((out == 7.0).all())
