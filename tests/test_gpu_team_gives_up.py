"""A one-launch solve whose waits reach their bound: every workgroup leaves, and the launched kernels finish the
solve from what x holds.  The bound is set from the host: 0 ends the first wait of every workgroup; a few polls
end waits anywhere in the solve, so that x is left from workgroups at different iterations."""

import pytest
import torch

from finite_elements_amd import _hip, device
from tests.test_gpu_team import _problem

pytestmark = pytest.mark.gpu

SYSTEMS = [('tet_elastic', 4, False), ('tri_elastic', (40, 10), True), ('tet_elastic', 13, False),
           ('tri_magnetic', (255, 255), False), ('tet_elastic', 32, True), ('tet_elastic', 41, False)]


@pytest.fixture
def spins(ctx):
    def set_spins(n):
        _hip.call('fe_pcg_set_spins', ctx.h, n)
    yield set_spins
    set_spins(_hip.FE_PCG_SPINS)


def _solver(ctx, kind, size, shuffled, precision, two_level=False):
    s, fixed, rng = _problem(kind, size, shuffled)
    mask, g = s.dirichlet(fixed)
    coarse = s.coarse_space(fixed) if two_level else None
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)), coarse=coarse)
    return s.solver(KD, 'two_level' if two_level else 'block_jacobi', precision, coarse=coarse), KD, b


@pytest.mark.parametrize('kind,size,shuffled', SYSTEMS)
def test_first_wait(ctx, spins, kind, size, shuffled):
    """Nothing was done: the launched kernels' bits, whatever the start."""
    precision = 'mixed' if size == 41 else 'fp64'
    print(f'first wait {kind} {size} {precision}', flush=True)
    solver, KD, b = _solver(ctx, kind, size, shuffled, precision)
    x0 = torch.rand_like(b)
    want = solver.solve(b, x=x0.clone(), tol=1e-9, max_iter=60, profile=True)
    spins(0)
    got = solver.solve(b, x=x0.clone(), tol=1e-9, max_iter=60)
    assert got[1]['path'] == _hip.FE_PCG_LEFT
    assert got[1]['iterations'] == want[1]['iterations'] and torch.equal(got[0], want[0])


@pytest.mark.parametrize('two_level', [False, True])
@pytest.mark.parametrize('kind,size,shuffled', SYSTEMS)
def test_any_wait(ctx, spins, kind, size, shuffled, two_level):
    precision = 'mixed' if size == 41 else 'fp64'
    print(f'any wait {kind} {size} {precision} {two_level}', flush=True)
    solver, KD, b = _solver(ctx, kind, size, shuffled, precision, two_level)
    tol = 1e-9
    for n in (0, 1, 2, 5, 20):
        spins(n)
        x, info = solver.solve(b, tol=tol)
        assert info['path'] in (_hip.FE_PCG_ONE_LAUNCH, _hip.FE_PCG_LEFT)
        assert n > 0 or info['path'] == _hip.FE_PCG_LEFT
        assert info['status'] == 0 and info['relres'] <= tol
        assert float((b - device.spmv(KD, x)).norm()) <= 1.001 * tol * float(b.norm())


def test_bound_is_checked(ctx):
    with pytest.raises(ValueError):
        _hip.call('fe_pcg_set_spins', ctx.h, -1)
