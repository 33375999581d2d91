"""The pattern in another node order (the two-level solve's, by aggregates) against a dense permutation."""

import numpy as np
import pytest

from finite_elements_amd.device import order_pattern, pad_pattern


@pytest.mark.parametrize('n,seed', [(1, 0), (2, 1), (17, 2), (64, 3)])
def test_order_pattern_is_the_permuted_matrix(n, seed):
    rng = np.random.default_rng(seed)
    dense = rng.random((n, n)) < 0.3
    dense |= dense.T | np.eye(n, dtype=bool)
    vals = rng.standard_normal((n, n)) * dense
    rows, cols = np.nonzero(dense)
    bptr = np.concatenate([[0], np.cumsum(dense.sum(axis=1))])
    order = rng.permutation(n)
    optr, ocol, src = order_pattern(bptr, cols, order)
    got = np.zeros((n, n))
    orow = np.repeat(np.arange(n), np.diff(optr))
    got[orow, ocol] = vals[rows, cols][src]
    assert np.array_equal(got, vals[np.ix_(order, order)])
    # padded: every row a multiple of four blocks, the additions pointing at the row itself
    pptr, pcol, psrc = pad_pattern(optr, ocol, 4)
    assert np.all(np.diff(pptr) % 4 == 0) and np.array_equal(pcol[psrc >= 0], ocol)
    assert np.array_equal(pcol[psrc < 0], np.repeat(np.arange(n), np.diff(pptr))[psrc < 0])
