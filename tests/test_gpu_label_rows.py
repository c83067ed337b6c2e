"""Rows of scores of every length and alignment: the first maximum, as torch.argmax."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [1, 3, 19, 20, 21, 40, 44])
def test_labels_take_the_first_maximum(C):
    from sparseconvnet import SCN as S

    rng = np.random.default_rng(C)
    pts = torch.from_numpy(np.stack([np.arange(777), np.zeros(777), np.zeros(777)], 1).astype(np.int64))
    score = torch.from_numpy(rng.integers(0, 4, (777, C)).astype(np.float32))  # (many ties)
    t = S.Result_3()
    t.set(pts, score)
    assert torch.equal(t.multiQuery(pts), torch.from_numpy(score.numpy().argmax(1)))
