"""The inverse of the coarse operator at the edges of its blocking: orders below, at and above a block of 16 or
64, one panel and several (an odd and an even number of them), dense and block-diagonal, and the block-diagonal
correction with it."""

import numpy as np
import pytest

from finite_elements_amd import meshgen
from oracle import coarse as oc
from tests.test_gpu_coarse import _host_matrix, _setup

pytestmark = pytest.mark.gpu


def _check(inv, inv32, A):
    ref = np.linalg.inv(A)
    err = np.abs(inv - ref).max() / np.abs(ref).max()
    assert err <= 1e-12 * np.linalg.cond(A)
    assert np.array_equal(inv, inv.T)
    assert np.array_equal(inv32, inv.astype(np.float32))


# (mesh, aggregate size) -> coarse DOFs
@pytest.mark.parametrize('n,target,order', [(10, 1000, 1), (10, 16, 9), (10, 8, 16), (20, 8, 49), (32, 17, 64),
                                            (20, 4, 100), (21, 4, 121), (40, 8, 196), (40, 4, 400)])
def test_inverse_orders(ctx, n, target, order):
    pr = meshgen.magnetostatic_2d(n=n)
    s, KD, _, dc = _setup(pr, target)
    assert dc.host.n_coarse == order
    ld = dc.ld
    A = dc.operator(KD, invert=False)[0].cpu().numpy().reshape(ld, ld)
    inv, inv32 = dc.operator(KD, invert=True)
    inv = inv.cpu().numpy().reshape(ld, ld)
    assert np.array_equal(inv[order:, order:], np.eye(ld - order)) and not inv[:order, order:].any()
    _check(inv[:order, :order], inv32.cpu().numpy().reshape(ld, ld)[:order, :order], A[:order, :order])
    if order <= 128:  # the same space as one segment's block
        seg = s.coarse_space(pr.fixed_dofs, target, node_offsets=[0, len(pr.coords)], max_block=128)
        k = seg.host.n_coarse
        A = seg.operator(KD, invert=False)[0].cpu().numpy()[:k * k].reshape(k, k)
        inv, inv32 = seg.operator(KD, invert=True)
        _check(inv.cpu().numpy()[:k * k].reshape(k, k), inv32.cpu().numpy()[:k * k].reshape(k, k), A)
        ref, P = oc.coarse_operator(seg.host, _host_matrix(KD))
        r = np.random.default_rng(order).standard_normal(P.shape[0])
        want = P @ np.linalg.solve(ref, P.T @ r)
        u = s.ctx.tensor(np.zeros(P.shape[0]))
        seg.apply(inv, s.ctx.tensor(r), u)
        assert np.abs(u.cpu().numpy() - want).max() <= 1e-10 * np.abs(want).max()
