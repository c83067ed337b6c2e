"""Weights packed by insc_conv_pack_weights are read as they are: a call with them launches the layer's kernel alone and
takes no scratch memory, so it can be captured, and they may fill the 4 GB that a kernel addresses."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
I64 = ctypes.c_int64


def call(x, wp, n_out, stream, raw=None):
    from sparseconvnet._lib import lib, ptr

    out = torch.full((x.shape[0], n_out), 7.0, device="cuda")
    run = lambda: lib.insc_conv_nbr(ptr(x), I64(x.shape[1]), I64(x.shape[0]), ptr(out), I64(n_out), raw, wp, None, None, 1, None,
                                    None, I64(x.shape[0]), x.shape[1], n_out, None, stream)
    return out, run


def packed(W):
    from sparseconvnet._lib import ensure_init, lib, ptr, stream_ptr

    ensure_init(0)
    wp = torch.empty(lib.insc_conv_packed_floats(1, *W.shape), device="cuda")
    lib.insc_conv_pack_weights(ptr(W), 1, W.shape[0], W.shape[1], ptr(wp), stream_ptr())
    return wp


def test_a_call_takes_no_memory():
    from sparseconvnet._lib import ptr

    x = torch.randn(40, 4096, device="cuda")
    W = torch.randn(4096, 4096, device="cuda") * 0.02
    wp = packed(W)
    hip = ctypes.CDLL("libamdhip64.so")
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0  # (one whose scratch memory nothing has asked for yet)
    out, run = call(x, ptr(wp), 4096, stream)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    run()
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == before
    ref = x.double() @ W.double()
    assert ((out - ref).abs().max() <= 1e-5 * ref.abs().max()).item()


@pytest.mark.parametrize("Cin,Cout", [(16, 16), (48, 96), (96, 40)])
def test_a_call_can_be_captured(Cin, Cout):
    from sparseconvnet._lib import ptr, stream_ptr

    x = torch.randn(777, Cin, device="cuda")
    W = torch.randn(Cin, Cout, device="cuda")
    wp = packed(W)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, run = call(x, ptr(wp), Cout, stream_ptr())
        run()
    for i in range(4):
        x.normal_()
        graph.replay()
        want, run = call(x, ptr(wp), Cout, stream_ptr())
        run()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and want.abs().max().item() > 0


@pytest.mark.parametrize("raw", [False, True])
def test_weights_of_3_gb(raw):
    """More than split weights may take (their 4 GB end at 2.86e9 bytes of packed ones)."""
    from sparseconvnet._lib import lib, ptr, stream_ptr

    C = 27520
    assert lib.insc_conv_split_floats(1, C, C) * 4 > 1 << 32 > lib.insc_conv_packed_floats(1, C, C) * 4
    x = torch.randn(33, C, device="cuda")
    W = torch.randn(C, C, device="cuda") * 0.01
    wp = None if raw else packed(W)
    out, run = call(x, None if raw else ptr(wp), C, stream_ptr(), ptr(W) if raw else None)
    run()
    for a in range(0, C, 5504):
        ref = x.double() @ W[:, a:a + 5504].double()
        assert ((out[:, a:a + 5504] - ref).abs().max() <= 1e-5 * ref.abs().max()).item()
    # (sums that are formed again read the same tiles)
    rows = out.clone()
    x[5, C - 7] = float("inf")
    run()
    assert torch.equal(out[5], torch.sign(W[C - 7]) * float("inf"))
    rows[5] = out[5]
    assert torch.equal(out, rows)
