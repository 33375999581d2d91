"""``upload``: several arrays in one copy hold what an upload each would."""

import numpy as np
import pytest
import torch

from finite_elements_amd import device
from finite_elements_amd.device import Context


@pytest.mark.parametrize('limit', [0, 64, 64 * 1024])
def test_packed_uploads(limit, monkeypatch):
    ctx = Context.__new__(Context)
    ctx.torch_device = torch.device('cpu')
    monkeypatch.setattr(device, 'PACK_BYTES', limit)
    rng = np.random.default_rng(0)
    arrays = [np.arange(5, dtype=np.int32), None, np.zeros(0, np.int16), rng.random((3, 4))[:, 1],
              rng.random((100, 200)), np.arange(12).reshape(3, 4).T, np.ones(3, np.uint8), np.zeros((0, 3), np.int32),
              np.arange(16, dtype=np.int64), np.arange(7, dtype=np.int16)]
    got = device.upload(ctx, *arrays)
    assert len(got) == len(arrays) and device.upload(ctx) == []
    for a, t in zip(arrays, got):
        if a is None:
            assert t is None
            continue
        want = ctx.tensor(a)
        assert t.dtype == want.dtype and t.is_contiguous() and torch.equal(t, want)
        assert t.data_ptr() % 16 == 0
