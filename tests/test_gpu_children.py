"""Children's update matrices pulled into their parent's panel and update matrix,
at the edges of the kernels' tiles: 16 and 32 columns of a narrow panel, tiles of
64 and 128 rows, no rows below, one to six children.  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H

pytestmark = pytest.mark.gpu


def nested(nc, mc, nr, leaves, rng):
    """Two middle blocks of mc columns, each with `leaves` leaf blocks of nc
    columns that reach every other row of it and of the nr root rows (children whose
    rows are a strict subset of their parent's); the middle blocks reach all of the
    root.  Diagonally dominant."""
    per = leaves * nc + mc
    n = 2 * per + nr
    a = np.zeros((n, n))
    root = slice(2 * per, n)
    for m in range(2):
        m0 = m * per
        mid = np.arange(m0 + leaves * nc, m0 + per)
        a[np.ix_(mid, mid)] = rng.standard_normal((mc, mc))
        a[root, mid] = rng.standard_normal((nr, mc))
        for k in range(leaves):
            b = np.arange(m0 + k * nc, m0 + (k + 1) * nc)
            rows = np.concatenate([mid[k % 2::2], np.arange(2 * per, n)[k % 2::2]])
            a[np.ix_(b, b)] = rng.standard_normal((nc, nc))
            a[np.ix_(rows, b)] = rng.standard_normal((len(rows), nc))
    a[root, root] = rng.standard_normal((nr, nr))
    a = np.tril(a, -1)
    a = a + a.T
    a[np.arange(n), np.arange(n)] = np.abs(a).sum(1) + 1.0
    return a


def csr(a):
    mask = a != 0.0
    rp = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    return rp, np.nonzero(mask)[1].astype(np.int32), a[mask]


@pytest.mark.parametrize("nc,mc,nr,leaves",
                         [(1, 2, 1, 1), (7, 15, 40, 2), (16, 16, 63, 3), (17, 17, 64, 4),
                          (16, 31, 65, 5), (32, 32, 127, 6), (32, 32, 128, 3), (32, 32, 129, 2),
                          (20, 33, 64, 3), (33, 32, 200, 4), (33, 129, 65, 3),
                          (40, 512, 129, 2), (40, 513, 128, 3), (24, 530, 300, 6),
                          (8, 20, 260, 150)])   # more tiles than the chip holds at once
def test_children_edges(nc, mc, nr, leaves):
    rng = np.random.default_rng(nc * 1000 + nr + leaves)
    a = nested(nc, mc, nr, leaves, rng)
    n = len(a)
    rp, ci, v = csr(a)
    c = H.Cholesky(rp, ci)
    for _ in range(2):   # the second factorization finds the first one's update matrices
        assert c.factor(v) == -1
        b = rng.standard_normal(n)
        x = c.solve(b)
        # backward error of a Cholesky solve is a small multiple of n eps; the
        # matrix is diagonally dominant with a condition number below 2 n
        assert np.linalg.norm(a @ x - b) <= 8 * n * np.finfo(float).eps * (
            np.linalg.norm(a, np.inf) * np.linalg.norm(x) + np.linalg.norm(b))
        assert np.linalg.norm(x - np.linalg.solve(a, b)) <= 1e-10 * np.linalg.norm(x)
    # not positive definite in a leaf, and in a middle block
    for at in (0, 2 * leaves * nc + mc + mc // 2):
        w = a.copy()
        w[at, at] = -w[at, at]
        assert c.factor(csr(w)[2]) != -1
    c.close()
