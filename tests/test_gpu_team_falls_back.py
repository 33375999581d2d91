"""A two-level solve that the one launch does not end goes on in the launched kernels in its own precision,
with their bits, and a system whose columns do not fit is not tried again."""

import ctypes

import numpy as np
import pytest
import torch

from finite_elements_amd import _hip, device
from finite_elements_amd.coarse import CoarseSpace
from tests.test_gpu_team import _hub, _problem

pytestmark = pytest.mark.gpu


def _fans(ctx, spokes=4000, fans=4):
    """Graph Laplacian (plus a half) of fans that share a centre, their hubs being nodes 0, 1, ... and one
    aggregate: the workgroup of the hubs' rows reads all other 16,000 rows, more than fit in its LDS (about
    6,300 in FP64, 11,200 in FP32)."""
    xy, fan = _hub(spokes)
    coords = np.concatenate([1e-3 * np.arange(fans)[:, None] * [[1.0, 0.0]]] + [xy[1:]] * fans)
    conn = np.concatenate([np.where(fan == 0, k, fan + fans - 1 + spokes * k) for k in range(fans)]).astype(np.int32)
    pat = device.Pattern(conn, 2, coords.shape[0])
    graph = device.DeviceGraph(ctx, pat)
    rows = np.repeat(np.arange(pat.n_nodes), np.diff(pat.bptr))
    vals = np.zeros((4, pat.nnzb))
    vals[0] = vals[3] = np.where(pat.bcol == rows, 0.5 + np.diff(pat.bptr)[rows], -1.0)
    KD = device.BsrMatrix(graph, ctx.tensor(vals.reshape(-1)), 2, _hip.FE_LAYOUT_PLANES)
    coarse = device.DeviceCoarse(ctx, CoarseSpace(coords, pat.bptr, pat.bcol, 2, target=200))
    return KD, coarse, ctx.tensor(np.random.default_rng(1).standard_normal(KD.n))


@pytest.mark.parametrize('mixed', [False, True])
def test_wide_rows(ctx, mixed):
    print(f'wide two-level mixed={mixed}', flush=True)
    KD, coarse, b = _fans(ctx)
    solver = device.PcgSolver(KD, 'block_jacobi', mixed=mixed, coarse=coarse)
    assert solver.ordered
    x0 = torch.rand_like(b)
    got = solver.solve(b, x=x0.clone(), tol=1e-9)
    want = solver.solve(b, x=x0.clone(), tol=1e-9, profile=True)
    assert got[1]['path'] == _hip.FE_PCG_WIDE and got[1]['status'] == 0
    for key in ('iterations', 'reliable_updates', 'relres', 'fallbacks'):
        assert got[1][key] == want[1][key], key
    assert torch.equal(got[0], want[0])
    again = solver.solve(b, x=x0.clone(), tol=1e-9)
    assert again[1]['path'] == _hip.FE_PCG_LAUNCHED and torch.equal(again[0], want[0])
    assert not device.PcgSolver(KD, 'block_jacobi', mixed=mixed, coarse=coarse).ordered
    assert device.PcgSolver(KD, 'block_jacobi', mixed=not mixed, coarse=coarse).ordered


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_waits_at_their_bound(ctx, precision):
    print(f'two-level bound {precision}', flush=True)
    s, fixed, rng = _problem('tet_elastic', 13, True)
    mask, g = s.dirichlet(fixed)
    coarse = s.coarse_space(fixed)
    KD, b = s.prepare(s.stiffness_bsr(), mask, g, ctx.tensor(rng.standard_normal(s.n)), coarse=coarse)
    solver = s.solver(KD, 'two_level', precision, coarse=coarse)
    want = solver.solve(b, tol=1e-9, profile=True)
    try:
        _hip.call('fe_pcg_set_spins', ctx.h, 0)
        got = solver.solve(b, tol=1e-9)
    finally:
        _hip.call('fe_pcg_set_spins', ctx.h, _hip.FE_PCG_SPINS)
    assert got[1]['path'] == _hip.FE_PCG_LEFT
    assert got[1]['iterations'] == want[1]['iterations'] and torch.equal(got[0], want[0])
    assert solver.solve(b, tol=1e-9)[1]['path'] == _hip.FE_PCG_ONE_LAUNCH


@pytest.mark.parametrize('mixed', [False, True])
def test_finished_in_the_call(ctx, mixed):
    """fe_pcg_coarse_ordered finishes such a solve itself, in FP64."""
    print(f'ordered entry mixed={mixed}', flush=True)
    KD, coarse, b = _fans(ctx)
    solver = device.PcgSolver(KD, 'block_jacobi', mixed=mixed, coarse=coarse)
    x, opts, stats, nbytes = torch.zeros_like(b), solver._opts(1e-9, 2000), _hip.FePcgStats(), ctypes.c_int64()
    a, it, c = KD.struct(), solver.A32.struct(), coarse.struct()
    ref = ctypes.byref
    _hip.call('fe_pcg_coarse_workspace', ctx.h, ref(a), ref(c), ref(opts), ref(nbytes))
    work = torch.empty(nbytes.value, dtype=torch.uint8, device=b.device)
    p = device._vp
    _hip.call('fe_pcg_coarse_ordered', ctx.h, ref(a), ref(it), p(solver.M64), p(solver.M32), ref(c), p(solver.Ainv64),
              p(b), p(x), p(work), work.numel(), ref(opts), ref(stats))
    assert stats.status == 0 and stats.relres <= 1e-9 and solver._path() == _hip.FE_PCG_WIDE
    assert float((b - device.spmv(KD, x)).norm()) <= 1.001e-9 * float(b.norm())
