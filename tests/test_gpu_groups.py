"""Inverses of groups of diagonal blocks and the sweeps through them, at the edges of
blocks (128 columns), groups (512) and items (64 rows; 16 to 128 columns against 1024
to 128 rows).  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H

pytestmark = pytest.mark.gpu


def two_level(nc, nr, rng):
    """Two dense blocks of nc columns, coupled to the same nr trailing rows.
    Diagonally dominant."""
    n = 2 * nc + nr
    a = rng.standard_normal((n, n))
    a[nc:2 * nc, :nc] = 0.0
    a = np.tril(a, -1)
    a = a + a.T
    a[np.arange(n), np.arange(n)] = np.abs(a).sum(1) + 1.0
    return a


@pytest.mark.parametrize("nc,nr", [(33, 63), (64, 65), (127, 128), (128, 129), (129, 256),
                                   (256, 257), (257, 300), (384, 511), (385, 512), (511, 513),
                                   (512, 600), (513, 64), (640, 1023), (1024, 130), (1025, 1),
                                   (1100, 1100)])
def test_group_edges(nc, nr):
    rng = np.random.default_rng(nc * 1000 + nr)
    a = two_level(nc, nr, rng)
    n = len(a)
    rp = np.concatenate([[0], np.cumsum((a != 0.0).sum(1))]).astype(np.int32)
    ci = np.nonzero(a)[1].astype(np.int32)
    c = H.Cholesky(rp, ci)
    for scale in (1.0, 3.0):   # the second factorization finds the first one's inverses
        assert c.factor(scale * a[a != 0.0]) == -1
        b = rng.standard_normal(n)
        x = c.solve(b)
        # backward error of a Cholesky solve is a small multiple of n eps; the
        # matrix is diagonally dominant with a condition number below 2 n
        assert np.linalg.norm(scale * (a @ x) - b) <= 8 * n * np.finfo(float).eps * (
            scale * np.linalg.norm(a, np.inf) * np.linalg.norm(x) + np.linalg.norm(b))
        assert np.linalg.norm(x - np.linalg.solve(scale * a, b)) <= 1e-10 * np.linalg.norm(x)
    c.close()
