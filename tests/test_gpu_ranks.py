"""Kernels that rank rows by wavefronts - radix passes, tile plans and their schedules, frames in one workgroup per scale -
at the edges of wavefronts, rounds and blocks."""
import ctypes

import numpy as np
import pytest
import torch

import test_gpu_primitives as primitives

pytestmark = pytest.mark.gpu
I64 = ctypes.c_int64
S = primitives.S


# a round of a wavefront, a wavefront's share of a block, a block, more blocks than counts in flight (32)
@pytest.mark.parametrize("n", [63, 65, 511, 512, 513, 2049, 65 * 1024, 66 * 1024 + 1])
def test_sort_edges(S, n):
    primitives.test_sort_stable(S, n, 16)


# frames of 256, second ones of 320, 1024, 1025 and 16383 points: rounds of 1024 rows, up to the last workgroup that ranks alone
@pytest.mark.parametrize("P", [256, 820, 821, 13107])
def test_frame_edges(S, P):
    primitives.test_insert_at_all_scales_equals_the_scale_by_scale_chain(S, P)


# one tile and less, a last group of one to four, a block of positions, more tiles than one round of the schedule (8 x 1024)
@pytest.mark.parametrize("n,listed", [(1, False), (31, True), (33, False), (129, True), (256, False), (257, True), (2049 * 32, True),
                                      (8193 * 32 + 5, False)])
def test_plan_and_schedule(S, n, listed):
    from sparseconvnet._lib import lib, ptr, stream_ptr

    g = torch.Generator(device="cuda").manual_seed(n)
    density = torch.rand((n, 1), generator=g, device="cuda") ** 4  # (tiles of many classes)
    nbr = torch.where(torch.rand((n, 27), generator=g, device="cuda") < density * 0.3,
                      torch.randint(0, n, (n, 27), generator=g, device="cuda"), -1).to(torch.int32)
    order = torch.randperm(n, generator=g, device="cuda").to(torch.int32) if listed else None
    nt = -(-n // 32)
    ld = nt * 32 + 64
    plan = torch.full((27, ld), -9, dtype=torch.int32, device="cuda")
    tmask = torch.full((ld // 32,), -9, dtype=torch.int32, device="cuda")
    sched = torch.full((ld // 32 + ld // 128 + 1,), -9, dtype=torch.int32, device="cuda")
    lib.insc_plan_build(ptr(nbr), None if order is None else ptr(order), None, I64(n), I64(ld), ptr(plan), ptr(tmask), ptr(sched),
                        stream_ptr())
    want = torch.full((nt * 32, 27), -1, dtype=torch.int32, device="cuda")
    want[:n] = nbr if order is None else nbr[order.long()]
    assert torch.equal(plan[:, :nt * 32], want.T) and bool((plan[:, nt * 32:] == -9).all())
    used = (want.view(nt, 32, 27) >= 0).any(1)
    assert torch.equal(tmask[:nt], (used.int() << torch.arange(27, device="cuda")).sum(1).int())
    groups = torch.cat([used, used.new_zeros((-nt % 4, 27))]).view(-1, 4, 27).any(1)
    for got, masks in ((sched[:nt], used), (sched[ld // 32:ld // 32 + len(groups)], groups)):
        assert torch.equal(got.sort().values, torch.arange(len(masks), dtype=torch.int32, device="cuda"))
        assert bool((masks.sum(1)[got.long()].diff() <= 0).all())
