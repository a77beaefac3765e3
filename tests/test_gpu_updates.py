"""Trailing updates in one launch or split over two streams, in 32-row or larger tiles:
one dense supernode around the tile counts where the launch changes (7, 8, 10 and 11
block columns after the first step).  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [129, 1023, 1024, 1025, 1408, 1409, 1537])
def test_update_launch_edges(n):
    rng = np.random.default_rng(n)
    a = np.tril(rng.standard_normal((n, n)), -1)
    a = a + a.T
    a[np.arange(n), np.arange(n)] = np.abs(a).sum(1) + 1.0
    c = H.Cholesky(np.arange(n + 1, dtype=np.int32) * n,
                   np.tile(np.arange(n, dtype=np.int32), n))
    b = rng.standard_normal(n)
    assert c.factor(a.ravel()) == -1
    x = c.solve(b)
    # backward error of a Cholesky solve is a small multiple of n eps
    assert np.linalg.norm(a @ x - b) <= 8 * n * np.finfo(float).eps * (
        np.linalg.norm(a, np.inf) * np.linalg.norm(x) + np.linalg.norm(b))
    # the failing pivot is found in the column where it is, after every update
    bad = a.copy()
    bad[n - 1, n - 1] = -1.0
    assert c.factor(bad.ravel()) == n - 1
    c.close()
