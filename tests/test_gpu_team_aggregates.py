"""The one-launch two-level solve on meshes whose aggregates are cut down by the domain's edge: bins of one or
two nodes, or of nodes on a line, leave some rigid-body modes dependent up to rounding, and their columns of T
reach 1e8.  The launched kernels are the reference."""

import numpy as np
import pytest
import torch

from finite_elements_amd import device, meshgen
from finite_elements_amd.system import FESystem

pytestmark = pytest.mark.gpu


def _round_part(kind, n):
    """The cells of a grid whose centre lies in a ball (disc), with the nodes moved off the grid."""
    coords, conn = meshgen.kuhn_tets(n) if kind == 'tet_elastic' else meshgen.structured_tri(n, n)
    conn = conn[((coords[conn].mean(axis=1) - 0.5) ** 2).sum(axis=1) < 0.25]
    used = np.unique(conn)
    new = np.full(coords.shape[0], -1)
    new[used] = np.arange(used.size)
    rng = np.random.default_rng(0)
    return coords[used] + 0.1 / n * rng.standard_normal((used.size, coords.shape[1])), new[conn].astype(np.int32)


# (kind, cells, nodes per aggregate, nodes left free in every other aggregate or None)
PARTS = [('tet_elastic', 12, 12, None), ('tet_elastic', 20, 100, None), ('tet_elastic', 20, 100, 1),
         ('tet_elastic', 27, 60, 2), ('tri_elastic', 60, 30, 1), ('tri_elastic', 120, 60, 1)]


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('kind,n,target,free', PARTS)
def test_dependent_modes(ctx, kind, n, target, free, precision):
    print(f'dependent modes {kind} {n} {target} {free} {precision}', flush=True)
    coords, conn = _round_part(kind, n)
    d, ne = coords.shape[1], conn.shape[0]
    rng = np.random.default_rng(1)
    s = FESystem(kind, coords, conn, {'E': np.exp(0.3 * rng.standard_normal(ne)), 'nu': np.full(ne, 0.3),
                                      'thickness': np.ones(ne)}, plane_mode=2 if d == 2 else 0)
    held = np.flatnonzero(coords[:, -1] < 0.1)
    if free is not None:  # hold all but `free` nodes of every eighth aggregate
        cs = s.coarse_space((held[:, None] * d + np.arange(d)).ravel(), target=target).host
        held = np.union1d(held, np.concatenate(
            [cs.agg_nodes[cs.agg_ptr[g] + free:cs.agg_ptr[g + 1]] for g in range(0, cs.n_agg, 8)]))
    fixed = (held[:, None] * d + np.arange(d)).ravel()
    mask, g = s.dirichlet(fixed)
    coarse = s.coarse_space(fixed, target=target)
    assert np.abs(coarse.host.T).max() > 1e6
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)), coarse=coarse)
    solver = s.solver(KD, 'two_level', precision, coarse=coarse)
    assert solver.ordered
    tol = 1e-9
    u, info = solver.solve(b, tol=tol)
    _, launched = solver.solve(b, tol=tol, profile=True)
    assert launched['status'] == 0
    assert info['status'] == 0 and info['relres'] <= tol
    assert info['iterations'] <= launched['iterations'] + 16 + launched['iterations'] // 8
    assert info['restarts'] <= launched['restarts'] and info['fallbacks'] <= launched['fallbacks']
    res = b - device.spmv(KD, u)
    assert float(res.norm()) <= 1.001 * tol * float(b.norm())
