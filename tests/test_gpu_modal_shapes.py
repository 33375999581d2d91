"""Edges of the Rayleigh-Ritz kernel and of the aggregate-wise residual pass: matrix orders around the
wavefront's pairs, entries far from 1, a basis without its full rank, and aggregates smaller and larger than
one pass of a workgroup."""

import numpy as np
import pytest
import torch

from finite_elements_amd import device, modal
from tests.test_gpu_modal import _check_pairs, _modal_system, _oracle_pencil, eigen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('r', [2, 3, 36, 63, 64, 65, 84, 95])
@pytest.mark.parametrize('scale', [1e-60, 1.0, 1e60])
def test_sym_eig_orders_and_scales(ctx, r, scale):
    rng = np.random.default_rng(100 + r)
    A = rng.standard_normal((2, r, r))
    A = A + A.transpose(0, 2, 1)
    A[1] = A[1] * np.outer(10.0 ** -np.linspace(0, 6, r), 10.0 ** -np.linspace(0, 6, r))  # graded
    w, V = modal.sym_eig(torch.as_tensor(A * scale, device=ctx.torch_device))
    w, V = w.cpu().numpy() / scale, V.cpu().numpy()
    for k in range(2):
        ref = np.linalg.eigvalsh(A[k])
        norm = max(1.0, np.abs(ref).max())
        assert np.max(np.abs(w[k] - ref)) <= 1e-13 * norm * r
        assert np.max(np.abs(A[k] @ V[k] - V[k] * w[k][None, :])) <= 1e-12 * norm * r
        assert np.max(np.abs(V[k].T @ V[k] - np.eye(r))) <= 1e-12 * r


@pytest.mark.parametrize('target', [8, 343])
@pytest.mark.parametrize('block', [4, 12, 32])
def test_lobpcg_aggregate_sizes(ctx, block, target):
    """343 nodes in more aggregates than residual chunks (runs of them) and in a single one (parts of it)."""
    pr, s = _modal_system(6, 5000)
    fixed, _ = s.dirichlet(pr.fixed_dofs)
    KD = device.apply_dirichlet(s.stiffness_bsr(), fixed)
    MD = device.apply_dirichlet(s.mass_bsr(), fixed)
    coarse = s.coarse_space(pr.fixed_dofs, target=target)
    chunks = -(-343 // 64)
    assert (coarse.struct().n_agg < chunks) == (target == 343)
    k = block - block // 4
    vals, vecs, info = modal.lobpcg(KD, MD, k, block=block, fixed=fixed, tol=1e-7, max_iter=3000, coarse=coarse)
    assert info['status'] == 0
    Ko, Mo = _oracle_pencil(pr)
    ref_vals, _ = eigen.smallest_clamped(Ko, Mo, pr.fixed_dofs, k)
    _check_pairs(vals[0], vecs[0].cpu().numpy(), Ko, Mo, pr.fixed_dofs, ref_vals)


def test_lobpcg_basis_without_full_rank(ctx):
    """A start block of converged vectors (residuals that add next to nothing to the basis) is accepted at
    once; one with a repeated column is refused as a breakdown."""
    pr, s = _modal_system(5, 5000)
    fixed, _ = s.dirichlet(pr.fixed_dofs)
    KD = device.apply_dirichlet(s.stiffness_bsr(), fixed)
    MD = device.apply_dirichlet(s.mass_bsr(), fixed)
    vals, vecs, info = modal.lobpcg(KD, MD, 8, block=8, fixed=fixed, tol=1e-9, max_iter=3000)
    assert info['status'] == 0
    X0 = vecs[0].cpu().numpy().copy()
    v2, _, i2 = modal.lobpcg(KD, MD, 8, block=8, fixed=fixed, tol=1e-7, max_iter=50, X0=X0)
    assert i2['status'] == 0 and int(i2['iterations'][0]) <= 2
    np.testing.assert_allclose(v2, vals, rtol=1e-8)
    X0[:, 5] = X0[:, 2]
    _, _, i3 = modal.lobpcg(KD, MD, 8, block=8, fixed=fixed, tol=1e-7, max_iter=50, X0=X0)
    assert i3['status'] != 0 and i3['failed'] == 1
