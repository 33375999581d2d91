"""Right-hand sides whose r . M r falls below the smallest normal number: scaling by a power of two changes no
rounding above that, so the solve takes the same course and its solution scales with it."""

import numpy as np
import pytest
import torch

from finite_elements_amd import meshgen
from finite_elements_amd.system import FESystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('profile', [False, True])  # the one-launch solve, the launched kernels
@pytest.mark.parametrize('problem', ['plate', 'cube'])
def test_subnormal_products(ctx, problem, profile):
    print(f'subnormal products {problem} {profile}', flush=True)
    pr = meshgen.cantilever_2d(40, 10) if problem == 'plate' else meshgen.cube_elasticity(n=8)
    s = FESystem(pr.kind, pr.coords, pr.conn, pr.materials, plane_mode=pr.plane_mode)
    mask, g = s.dirichlet(pr.fixed_dofs)
    f = ctx.tensor(np.random.default_rng(0).standard_normal(s.n))
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, f)
    solver = s.solver(KD, 'jacobi', 'fp64')
    tol = 1e-6
    x, want = solver.solve(b, tol=tol, profile=profile)
    assert want['status'] == 0
    # |b|^2 near 1e-292, so tol^2 |b|^2 and r . r stay normal; the diagonal of K is above 1e9, so r . M r
    # ends below 1e-313
    scale = 2.0 ** round(np.log2(1e-146 / float(b.norm())))
    xs, got = solver.solve(b * scale, tol=tol, profile=profile)
    assert got['status'] == 0 and got['relres'] <= tol
    # products of 1e-313 are rounded to 1e-11 of themselves: the course changes by an iteration or two at most
    assert abs(got['iterations'] - want['iterations']) <= 2
    assert torch.allclose(xs / scale, x, rtol=0, atol=1e-6 * float(x.abs().max()))
