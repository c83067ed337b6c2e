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
