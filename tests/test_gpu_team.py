"""The one-launch solve (a team of workgroups) against the launched kernels, bit for bit: the profiled solve
always runs the launched ones.  Sizes are at the edges of its rules: one tile, one workgroup of two
tiles, the last size of each workgroup shape and the first of the next, rows longer than one vector step,
columns scattered over the system, a row count that ends inside a tile."""

import numpy as np
import pytest
import torch

from finite_elements_amd import _hip, device, meshgen
from finite_elements_amd.system import FESystem

pytestmark = pytest.mark.gpu


def _hub(spokes):
    """A fan: `spokes` outer nodes around one node, whose row holds them all."""
    t = 2 * np.pi * np.arange(spokes) / spokes
    coords = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], axis=1)])
    i = 1 + np.arange(spokes)
    conn = np.stack([np.zeros(spokes, dtype=np.int64), i, 1 + i % spokes], axis=1)
    return coords, conn.astype(np.int32)


def _problem(kind, size, shuffled=False, seed=0):
    rng = np.random.default_rng(seed)
    if kind == 'tet_elastic':
        coords, conn = meshgen.kuhn_tets(size)
        held, d = np.flatnonzero(coords[:, 2] == 0.0), 3
    elif size == 'hub':
        coords, conn = _hub(300)
        held, d = np.arange(1, 40), 1 if kind == 'tri_magnetic' else 2
    else:
        coords, conn = meshgen.structured_tri(*size)
        held, d = np.flatnonzero(coords[:, 0] == 0.0), 1 if kind == 'tri_magnetic' else 2
    if shuffled:
        new = rng.permutation(coords.shape[0])
        old = np.argsort(new)
        coords, conn, held = coords[old], new[conn].astype(np.int32), np.sort(new[held])
    ne = conn.shape[0]
    mats = {'mu': np.exp(rng.standard_normal(ne))} if kind == 'tri_magnetic' else {
        'E': np.exp(0.3 * rng.standard_normal(ne)), 'nu': np.full(ne, 0.3), 'thickness': np.ones(ne)}
    fixed = (held[:, None] * d + np.arange(d)).ravel()
    return FESystem(kind, coords, conn, mats, plane_mode=0 if d != 2 else 2), fixed, rng


# (kind, size, shuffled): tiles of 128 rows with three DOF per node, 256 with one or two
SIZES = [('tet_elastic', 2, False), ('tet_elastic', 4, False), ('tet_elastic', 5, True),
         ('tet_elastic', 13, False), ('tet_elastic', 27, True), ('tet_elastic', 32, False),
         ('tri_magnetic', (3, 3), False), ('tri_magnetic', (16, 16), False), ('tri_magnetic', (31, 17), True),
         ('tri_magnetic', (255, 255), False), ('tri_magnetic', (256, 255), False),
         ('tri_magnetic', 'hub', False), ('tri_elastic', (5, 2), False), ('tri_elastic', (40, 10), True),
         ('tri_elastic', (100, 50), False), ('tri_elastic', (361, 181), True), ('tri_elastic', 'hub', False)]


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('precond', ['jacobi', 'block_jacobi'])
@pytest.mark.parametrize('kind,size,shuffled', SIZES)
def test_team_equals_launched_kernels(ctx, kind, size, shuffled, precond, precision):
    print(f'team {kind} {size} {shuffled} {precond} {precision}', flush=True)
    s, fixed, rng = _problem(kind, size, shuffled)
    mask, g = s.dirichlet(fixed)
    f = ctx.tensor(rng.standard_normal(s.n))
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, f)
    solver = s.solver(KD, precond, precision)
    x0 = ctx.tensor(rng.standard_normal(s.n)) * (1 - mask.double())
    for start in (None, x0):
        # enough iterations for a few reliable updates, few enough for the largest system
        got = solver.solve(b, x=None if start is None else start.clone(), tol=1e-9, max_iter=150)
        want = solver.solve(b, x=None if start is None else start.clone(), tol=1e-9, max_iter=150, profile=True)
        for key in ('iterations', 'reliable_updates', 'restarts', 'status', 'relres', 'relres_rec'):
            assert got[1][key] == want[1][key], key
        assert torch.equal(got[0], want[0])


@pytest.mark.parametrize('n,precision', [(41, 'mixed'), (50, 'mixed'), (51, 'mixed'), (41, 'fp64')])
def test_team_size_limits(ctx, n, precision):
    """Four tiles per workgroup (FP32), the last size that a team takes, and the sizes beyond."""
    print(f'team limits {n} {precision}', flush=True)
    s, fixed, rng = _problem('tet_elastic', n)
    mask, g = s.dirichlet(fixed)
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)))
    solver = s.solver(KD, 'block_jacobi', precision)
    got = solver.solve(b, tol=1e-9, max_iter=60)
    want = solver.solve(b, tol=1e-9, max_iter=60, profile=True)
    assert got[1]['iterations'] == want[1]['iterations'] and torch.equal(got[0], want[0])


def test_team_gives_way_when_its_columns_do_not_fit(ctx):
    """Three rows of 4,000 columns in one workgroup, whose u does not fit in its LDS: the launched kernels
    solve it.  (Graph Laplacians of three fans whose hubs are nodes 0, 1 and 2.)"""
    print('team overflow', flush=True)
    _, fan = _hub(4000)
    conn = np.concatenate([np.where(fan == 0, k, fan + 2 + 4000 * k) for k in range(3)]).astype(np.int32)
    pat = device.Pattern(conn, 2, 3 + 3 * 4000)
    graph = device.DeviceGraph(ctx, pat)
    rows = np.repeat(np.arange(pat.n_nodes), np.diff(pat.bptr))
    on = pat.bcol == rows
    vals = np.zeros((4, pat.nnzb))
    vals[0] = vals[3] = np.where(on, 0.5 + np.diff(pat.bptr)[rows], -1.0)
    KD = device.BsrMatrix(graph, ctx.tensor(vals.reshape(-1)), 2, _hip.FE_LAYOUT_PLANES)
    b = ctx.tensor(np.random.default_rng(1).standard_normal(KD.n))
    solver = device.PcgSolver(KD, 'block_jacobi')
    got = solver.solve(b, tol=1e-10)
    want = solver.solve(b, tol=1e-10, profile=True)
    assert got[1]['status'] == 0 and got[1]['iterations'] == want[1]['iterations']
    assert torch.equal(got[0], want[0])


def test_team_statuses(ctx):
    """Zero right-hand side, iteration limit and breakdown come out as from the launched kernels."""
    print('team statuses', flush=True)
    s, fixed, rng = _problem('tet_elastic', 6)
    mask, g = s.dirichlet(fixed)
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)))
    solver = s.solver(KD, 'jacobi', 'fp64')
    x, info = solver.solve(torch.zeros_like(b))
    assert info['status'] == 0 and info['iterations'] == 0 and not x.any()
    _, info = solver.solve(b, tol=1e-12, max_iter=5)
    assert info['status'] == _hip.FE_ERR_NOT_CONVERGED and info['iterations'] == 5
    KD.vals.neg_()
    solver = s.solver(KD, 'jacobi', 'fp64', M64=device.precond_setup(KD, 'jacobi').abs())
    _, info = solver.solve(b)
    assert info['status'] == _hip.FE_ERR_BREAKDOWN


# (kind, size, shuffled, nodes per aggregate): many aggregates in a tile, aggregates as long as a tile (their
# ends meet), tiles inside one aggregate, one tile, one workgroup of two tiles, several workgroup shapes
COARSE = [('tet_elastic', 3, False, 8), ('tet_elastic', 5, True, 30), ('tet_elastic', 7, False, 128),
          ('tet_elastic', 13, True, 1000), ('tet_elastic', 27, True, None), ('tet_elastic', 33, False, None),
          ('tri_magnetic', (15, 15), False, 256), ('tri_magnetic', (31, 17), True, 20),
          ('tri_magnetic', (127, 127), False, 256), ('tri_magnetic', (300, 300), False, None),
          ('tri_elastic', (9, 4), False, 12), ('tri_elastic', (40, 10), True, 81),
          ('tri_elastic', (120, 50), False, None), ('tri_elastic', (400, 200), False, None),
          ('tri_magnetic', (400, 400), True, None)]


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('kind,size,shuffled,target', COARSE)
def test_team_two_level(ctx, kind, size, shuffled, target, precision):
    """The two-level solve in the order of the aggregates: it reaches the tolerance on the true residual,
    in the launched kernels' iterations (the correction is carried by recurrence, so not bit for bit), and
    a second solve by the same solver gives the same bits."""
    print(f'team two-level {kind} {size} {shuffled} {target} {precision}', flush=True)
    s, fixed, rng = _problem(kind, size, shuffled)
    mask, g = s.dirichlet(fixed)
    coarse = s.coarse_space(fixed, target=target)
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)), coarse=coarse)
    solver = s.solver(KD, 'two_level', precision, coarse=coarse)
    assert solver.ordered
    tol = 1e-9
    u, info = solver.solve(b, tol=tol)
    assert info['status'] == 0 and info['relres'] <= tol and info['fallbacks'] == 0
    res = b - device.spmv(KD, u)
    assert float(res.norm()) <= 1.001 * tol * float(b.norm())
    _, launched = solver.solve(b, tol=tol, profile=True)
    assert launched['status'] == 0
    assert abs(info['iterations'] - launched['iterations']) <= 16 + launched['iterations'] // 8
    u2, info2 = solver.solve(b, tol=tol)
    assert info2['iterations'] == info['iterations'] and torch.equal(u, u2)
    # a start that already solves the system needs no iteration, and keeps its bits
    x, info = solver.solve(b, x=u.clone(), tol=2 * tol)
    assert info['iterations'] == 0 and torch.equal(x, u)


def test_team_two_level_beyond_its_sizes(ctx):
    """FP64 beyond 512 tiles and a coarse space beyond its limit go to the launched kernels."""
    print('team two-level limits', flush=True)
    s, fixed, _ = _problem('tet_elastic', 41)
    mask, g = s.dirichlet(fixed)
    coarse = s.coarse_space(fixed)
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.zeros(s.n), coarse=coarse)
    assert not s.solver(KD, 'two_level', 'fp64', coarse=coarse).ordered
    assert s.solver(KD, 'two_level', 'mixed', coarse=coarse).ordered
    s, fixed, rng = _problem('tri_magnetic', (60, 60))
    mask, g = s.dirichlet(fixed)
    coarse = s.coarse_space(fixed, target=2)
    assert coarse.n_coarse > 1536
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)), coarse=coarse)
    solver = s.solver(KD, 'two_level', 'fp64', coarse=coarse)
    assert not solver.ordered
    assert solver.solve(b, tol=1e-9)[1]['status'] == 0
