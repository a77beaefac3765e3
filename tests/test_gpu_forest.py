"""Small supernodes at the edges of the sweeps' items: one wave (fronts of 64
rows), a workgroup (256 rows at a time, up to 512), the top of the tree beyond
32 columns or 512 rows.  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H

pytestmark = pytest.mark.gpu


def arrow(nc, nr, leaves, rng):
    """`leaves` dense blocks of nc columns, each coupled to the same nr trailing
    rows: supernodes of nc columns on nr rows below a dense root.  Diagonally
    dominant."""
    n = leaves * nc + nr
    a = np.zeros((n, n))
    for k in range(leaves):
        b = slice(k * nc, (k + 1) * nc)
        a[b, b] = rng.standard_normal((nc, nc))
        a[leaves * nc:, b] = rng.standard_normal((nr, nc))
    t = slice(leaves * nc, n)
    a[t, t] = rng.standard_normal((nr, nr))
    a = np.tril(a, -1)
    a = a + a.T
    a[np.arange(n), np.arange(n)] = np.abs(a).sum(1) + 1.0
    return a


def csr(a):
    mask = a != 0.0
    rp = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    return rp, np.nonzero(mask)[1].astype(np.int32), a[mask]


@pytest.mark.parametrize("nc,nr", [(1, 1), (4, 28), (9, 55), (32, 32), (32, 33), (31, 225),
                                   (32, 225), (16, 300), (32, 480), (32, 481), (33, 20)])
def test_forest_edges(nc, nr):
    rng = np.random.default_rng(nc * 1000 + nr)
    a = arrow(nc, nr, 5, rng)
    rp, ci, v = csr(a)
    c = H.Cholesky(rp, ci)
    assert c.factor(v) == -1
    for _ in range(2):
        b = rng.standard_normal(len(a))
        x = c.solve(b)
        # backward error of a Cholesky solve is a small multiple of n eps; the
        # matrix is diagonally dominant with a condition number below 2 n
        n = len(a)
        assert np.linalg.norm(a @ x - b) <= 8 * n * np.finfo(float).eps * (
            np.linalg.norm(a, 2) * np.linalg.norm(x) + np.linalg.norm(b))
        assert np.linalg.norm(x - np.linalg.solve(a, b)) <= 1e-10 * np.linalg.norm(x)
    c.close()
