"""Tensors of one packed upload are independent for autograd: changing one in place leaves a graph that has
saved another usable."""

import numpy as np
import torch

from finite_elements_amd import device
from finite_elements_amd.device import Context


def test_in_place_change_of_a_neighbour():
    ctx = Context.__new__(Context)
    ctx.torch_device = torch.device('cpu')
    a, b, mask = device.upload(ctx, np.arange(10.0), np.ones(10), np.zeros(10, np.uint8))
    w = torch.ones(10, dtype=torch.float64, requires_grad=True)
    y = (a * w).sum()
    b.mul_(2.0)
    mask[3] = 1
    y.backward()
    assert torch.equal(w.grad, a) and torch.equal(b, torch.full((10,), 2.0, dtype=torch.float64))
    assert int(mask.sum()) == 1
    a.requires_grad_()
    assert a.is_leaf and not b.requires_grad
