"""Which systems the one-launch solve takes, and that it is what ran: at each workgroup shape's first and last
sizes, against the launched kernels (bit for bit without a coarse space; with one, the correction is
carried by recurrence, so by tolerance and iterations)."""

import ctypes

import pytest
import torch

from finite_elements_amd import _hip, device
from tests.test_gpu_team import COARSE, SIZES, _problem

pytestmark = pytest.mark.gpu

LAUNCHED, ONE_LAUNCH = _hip.FE_PCG_LAUNCHED, _hip.FE_PCG_ONE_LAUNCH


def _prepared(ctx, kind, size, shuffled=False, target=0):
    """(system, K_D, b, coarse space or None); target 0: no coarse space, None: the default one."""
    s, fixed, rng = _problem(kind, size, shuffled)
    mask, g = s.dirichlet(fixed)
    coarse = None if target == 0 else s.coarse_space(fixed, target=target)
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)), coarse=coarse)
    return s, KD, b, coarse


@pytest.mark.parametrize('kind,size,shuffled', SIZES)
def test_small_systems_run_in_one_launch(ctx, kind, size, shuffled):
    print(f'path {kind} {size} {shuffled}', flush=True)
    s, KD, b, _ = _prepared(ctx, kind, size, shuffled)
    for precond in ('jacobi', 'block_jacobi'):
        for precision in ('fp64', 'mixed'):
            solver = s.solver(KD, precond, precision)
            assert solver.solve(b, tol=1e-9, max_iter=20)[1]['path'] == ONE_LAUNCH
            assert solver.solve(b, tol=1e-9, max_iter=20, profile=True)[1]['path'] == LAUNCHED


@pytest.mark.parametrize('kind,size,shuffled,target', COARSE)
def test_small_two_level_systems_run_in_one_launch(ctx, kind, size, shuffled, target):
    print(f'path two-level {kind} {size} {shuffled} {target}', flush=True)
    s, KD, b, coarse = _prepared(ctx, kind, size, shuffled, target)
    for precision in ('fp64', 'mixed'):
        solver = s.solver(KD, 'two_level', precision, coarse=coarse)
        assert solver.solve(b, tol=1e-9)[1]['path'] == ONE_LAUNCH
        assert solver.solve(b, tol=1e-9, profile=True)[1]['path'] == LAUNCHED


# tiles of 128 rows (three DOF per node) or 256; 512 in FP64 and 1,024 in FP32 are the limits, and more than
# 512 tiles are four to a workgroup
LIMITS = [('tet_elastic', 39, 'fp64', True),            # 500 tiles
          ('tet_elastic', 40, 'fp64', False),           # 539
          ('tet_elastic', 41, 'mixed', True),           # 579, four tiles per workgroup
          ('tet_elastic', 49, 'mixed', True),           # 977
          ('tet_elastic', 50, 'mixed', False),          # 1,037
          ('tri_magnetic', (370, 370), 'mixed', True),  # 538
          ('tri_magnetic', (370, 370), 'fp64', False),
          ('tri_magnetic', (511, 511), 'mixed', True),  # 1,024
          ('tri_magnetic', (512, 511), 'mixed', False),
          ('tri_elastic', (520, 260), 'mixed', True),   # 532
          ('tri_elastic', (520, 260), 'fp64', False),
          ('tri_elastic', (723, 361), 'mixed', True)]   # 1,024, the last of them short


@pytest.mark.parametrize('precond', ['jacobi', 'block_jacobi'])
@pytest.mark.parametrize('kind,size,precision,taken', LIMITS)
def test_size_limits(ctx, kind, size, precision, taken, precond):
    print(f'limit {kind} {size} {precision} {precond}', flush=True)
    s, KD, b, _ = _prepared(ctx, kind, size)
    solver = s.solver(KD, precond, precision)
    got = solver.solve(b, tol=1e-9, max_iter=60)
    want = solver.solve(b, tol=1e-9, max_iter=60, profile=True)
    assert got[1]['path'] == (ONE_LAUNCH if taken else LAUNCHED) and want[1]['path'] == LAUNCHED
    for key in ('iterations', 'reliable_updates', 'restarts', 'status', 'relres', 'relres_rec'):
        assert got[1][key] == want[1][key], key
    assert torch.equal(got[0], want[0])


@pytest.mark.parametrize('kind,size,shuffled,precision', [
    ('tet_elastic', 39, False, 'fp64'), ('tet_elastic', 41, True, 'mixed'), ('tet_elastic', 49, False, 'mixed'),
    ('tri_magnetic', (511, 511), False, 'fp64'), ('tri_magnetic', (511, 511), True, 'mixed'),
    ('tri_elastic', (520, 260), True, 'fp64'), ('tri_elastic', (723, 361), False, 'mixed')])
def test_two_level_limits(ctx, kind, size, shuffled, precision):
    print(f'two-level limit {kind} {size} {shuffled} {precision}', flush=True)
    s, KD, b, coarse = _prepared(ctx, kind, size, shuffled, None)
    solver = s.solver(KD, 'two_level', precision, coarse=coarse)
    tol = 1e-9
    u, info = solver.solve(b, tol=tol)
    assert info['path'] == ONE_LAUNCH
    assert info['status'] == 0 and info['relres'] <= tol and info['fallbacks'] == 0
    assert float((b - device.spmv(KD, u)).norm()) <= 1.001 * tol * float(b.norm())
    _, launched = solver.solve(b, tol=tol, profile=True)
    assert launched['path'] == LAUNCHED and launched['status'] == 0
    assert abs(info['iterations'] - launched['iterations']) <= 16 + launched['iterations'] // 8


def test_empty_system(ctx):
    """A system without rows launches nothing, whatever ran before it."""
    s, KD, b, _ = _prepared(ctx, 'tri_elastic', (5, 2))
    solver = s.solver(KD, 'jacobi', 'fp64')
    assert solver.solve(b, tol=1e-9)[1]['path'] == ONE_LAUNCH
    empty = KD.struct()
    empty.n_brows = empty.nnzb = 0
    opts, stats, p = solver._opts(1e-9, 10), _hip.FePcgStats(), device._vp
    work = torch.empty(4096, dtype=torch.uint8, device=b.device)
    _hip.call('fe_pcg', ctx.h, ctypes.byref(empty), None, p(solver.M64), None, p(b), p(torch.zeros_like(b)), p(work),
              work.numel(), ctypes.byref(opts), ctypes.byref(stats))
    assert stats.status == 0 and solver._path() == LAUNCHED
