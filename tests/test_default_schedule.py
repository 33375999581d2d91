"""The default row-block schedule on both sides of the size where its ranges grow, and the assembly's bits there."""

import numpy as np
import pytest
import torch

from finite_elements_amd import meshgen
from finite_elements_amd.device import Pattern
from finite_elements_amd.system import FESystem


def _mesh(kind, n):
    if kind == 'tet_elastic':
        return meshgen.kuhn_tets(n)
    return meshgen.structured_tri(n, n, 1.0, 1.0)


# 8 ranges of 256 incidences per CU: 524,288 incidences, 24 n^3 of a cube and 6 n^2 of a square
@pytest.mark.parametrize('kind,n,cap', [('tet_elastic', 27, 192), ('tet_elastic', 28, 256),
                                        ('tri_magnetic', 295, 128), ('tri_magnetic', 296, 256)])
def test_default_ranges(kind, n, cap):
    coords, conn = _mesh(kind, n)
    pat = Pattern(conn, 3 if kind == 'tet_elastic' else 1, coords.shape[0])
    assert (pat.n_inc >= 8 * 256 * 256) == (cap == 256)
    blk, biggest = Pattern.schedule_for(pat.inc_ptr, cap)
    assert np.array_equal(blk, pat.blk) and biggest == pat.max_inc <= cap


@pytest.mark.gpu
@pytest.mark.parametrize('what', ['stiffness', 'mass'])
@pytest.mark.parametrize('kind,n,cap', [('tet_elastic', 28, 192), ('tri_elastic', 296, 128)])
def test_default_ranges_same_bits(ctx, kind, n, cap, what):
    coords, conn = _mesh(kind, n)
    rng = np.random.default_rng(n)
    mats = {'E': rng.uniform(1.0, 2.0, conn.shape[0]), 'nu': np.full(conn.shape[0], 0.3),
            'rho': np.full(conn.shape[0], 2.0), 'thickness': np.full(conn.shape[0], 0.5)}
    s = FESystem(kind, coords, conn, mats, plane_mode=2 if kind == 'tri_elastic' else 0)
    got = getattr(s, what)().clone()
    s.set_schedule(cap)
    assert torch.equal(got, getattr(s, what)())
