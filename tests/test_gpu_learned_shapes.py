"""Weight gradients of the learned preconditioner at node counts around the edges of the gradient kernel:
fewer nodes than one step of a wavefront, odd counts, and more than the grid takes in one pass."""

import ctypes

import numpy as np
import pytest
import torch

from finite_elements_amd import _hip, learned, meshgen
from oracle import gnn as ognn

pytestmark = pytest.mark.gpu


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


# (nx, ny) of a triangle mesh: 4, 9, 15, 35, 65, 8,255 and 66,049 nodes
@pytest.mark.parametrize('nx,ny,dof', [(1, 1, 1), (2, 2, 3), (2, 4, 2), (4, 6, 3), (4, 12, 1), (64, 126, 2),
                                       (256, 256, 1)])
def test_backward_matches_autograd(ctx, nx, ny, dof):
    from finite_elements_amd.system import FESystem
    print(f'gnn backward {nx}x{ny} dof {dof}', flush=True)
    coords, conn = meshgen.structured_tri(nx, ny)
    s = FESystem('tri_magnetic', coords, conn, {'mu': 1.0})
    n = coords.shape[0]
    rng = np.random.default_rng(nx * 1000 + ny)
    p = learned.init_params(dof, seed=2)
    p[-(dof * 32 + dof):] = rng.normal(0, 0.3, dof * 32 + dof)
    feat = rng.standard_normal((n, 8)).astype(np.float32)
    dlo = rng.standard_normal((n, dof)).astype(np.float32)
    t = ctx.tensor
    f_t, d_t, p_t = t(feat), t(dlo), t(p.astype(np.float32))
    acts, aggs, o = ctx.empty(3 * n * 32, torch.float32), ctx.empty(n * 72, torch.float32), ctx.empty(n * dof, torch.float32)
    binv, M = ctx.zeros(n * dof * dof), ctx.empty(n * dof * dof)
    g = s.graph
    _hip.call('fe_gnn_forward', ctx.h, n, dof, _vp(g.bptr), _vp(g.bcol), _vp(p_t), _vp(f_t), _vp(acts),
              _vp(aggs), _vp(binv), _vp(o), _vp(M))
    nb = ctypes.c_int64()
    _hip.call('fe_gnn_backward_workspace', n, ctypes.byref(nb))
    work = ctx.empty(nb.value, torch.float32)
    grad = ctx.zeros(p.size, torch.float32)
    _hip.call('fe_gnn_backward', ctx.h, n, dof, _vp(g.bptr), _vp(g.bcol), _vp(p_t), _vp(f_t), _vp(acts),
              _vp(aggs), _vp(d_t), _vp(work), _vp(grad))
    # the mean over the neighbours, without a loop over the nodes
    pat = s.pattern
    rows = np.repeat(np.arange(n), np.diff(pat.bptr))
    off = pat.bcol != rows
    deg = np.bincount(rows[off], minlength=n).astype(np.float64)
    avg = torch.sparse_coo_tensor(np.vstack([rows[off], pat.bcol[off]]), 1.0 / deg[rows[off]], (n, n),
                                  dtype=torch.float64)
    P = torch.tensor(p, dtype=torch.float64, requires_grad=True)
    ognn.forward(P, feat.astype(np.float64), avg, dof).backward(torch.as_tensor(dlo, dtype=torch.float64))
    ref, got = P.grad.numpy(), grad.cpu().numpy()
    # FP32 sums of at most 66,049 terms (unit roundoff 6e-8, random signs: about 2e-5 of the sum of
    # moduli), and a ReLU whose argument rounds across zero in a few of the nodes
    assert np.linalg.norm(got - ref) <= 1e-3 * np.linalg.norm(ref)
