"""Fronts with many small children, which get no index of their children's rows and take
their update matrices by extend-add, beside fronts with few.  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H
from test_gpu_children import csr

pytestmark = pytest.mark.gpu


def hub(mc, nr, leaves, rng):
    """Two middle blocks of mc columns coupled to all nr root rows, each with `leaves`
    one-column children that reach one of its columns and one or two root rows.
    Diagonally dominant."""
    per = leaves + mc
    n = 2 * per + nr
    a = np.zeros((n, n))
    root = np.arange(2 * per, n)
    for m in range(2):
        m0 = m * per
        mid = np.arange(m0 + leaves, m0 + per)
        a[np.ix_(mid, mid)] = rng.standard_normal((mc, mc))
        a[np.ix_(root, mid)] = rng.standard_normal((nr, mc))
        for k in range(leaves):
            a[mid[k % mc], m0 + k] = rng.standard_normal()
            a[rng.choice(root, 1 + k % 2), m0 + k] = rng.standard_normal()
    a[np.ix_(root, root)] = rng.standard_normal((nr, nr))
    a = np.tril(a, -1)
    a = a + a.T
    a[np.arange(n), np.arange(n)] = np.abs(a).sum(1) + 1.0
    return a


# twelve and 17 children: with an index; the others without
@pytest.mark.parametrize("mc,nr,leaves", [(20, 40, 12), (20, 40, 17), (20, 40, 18), (20, 150, 400), (32, 300, 700),
                                          (33, 129, 300), (140, 260, 900), (600, 200, 800)])
def test_hub(mc, nr, leaves):
    rng = np.random.default_rng(mc + nr + leaves)
    a = hub(mc, nr, leaves, rng)
    n = len(a)
    rp, ci, v = csr(a)
    c = H.Cholesky(rp, ci)
    for _ in range(2):   # the second factorization finds the first one's update matrices
        assert c.factor(v) == -1
        b = rng.standard_normal(n)
        x = c.solve(b)
        # backward error of a Cholesky solve is a small multiple of n eps; the matrix is
        # diagonally dominant with a condition number below 2 n
        assert np.linalg.norm(a @ x - b) <= 8 * n * np.finfo(float).eps * (
            np.linalg.norm(a, np.inf) * np.linalg.norm(x) + np.linalg.norm(b))
        assert np.linalg.norm(x - np.linalg.solve(a, b)) <= 1e-10 * np.linalg.norm(x)
    c.close()
