"""Backward errors of Cholesky solves with ill-conditioned fronts: the inverses that the
sweeps multiply with must not lose more than one condition number.  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H
from hykkt_amd.generator import GridPattern, ds_spread_schedule
from test_gpu_batch_engine import alone

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def backward_errors(a, vals, rp, ci, rng):
    """Normwise, residuals in extended precision; right-hand sides random and with
    random solutions."""
    c = H.Cholesky(rp, ci)
    assert c.factor(vals) == -1
    norm = np.abs(a).sum(1).max()
    out = []
    for k in range(6):
        b = rng.standard_normal(len(a))
        if k % 2:
            b = a @ b
        x = c.solve(b)
        r = np.asarray(b - a.astype(np.longdouble) @ x.astype(np.longdouble), float)
        out.append(np.linalg.norm(r) / (norm * np.linalg.norm(x) + np.linalg.norm(b)))
    c.close()
    return out


@pytest.mark.parametrize("n", [256, 300, 512, 1000])
def test_gaussian_kernel(n):
    """One dense supernode, condition number about 1e11.  With an inverse X of a group's
    triangle L as accurate as its own condition allows, y = X v errs by eps |X| |L| |y|:
    the solve's backward error is at most about eps cond(L)."""
    x = np.linspace(0.0, 1.0, n)
    a = np.exp(-200.0 * (x[:, None] - x) ** 2) + 1e-9 * np.eye(n)
    rp = (np.arange(n + 1) * n).astype(np.int32)
    ci = np.tile(np.arange(n), n).astype(np.int32)
    be = backward_errors(a, a.ravel(), rp, ci, np.random.default_rng(n))
    cond = np.linalg.cond(np.linalg.cholesky(a))
    print(f"{n}: backward errors {max(be):.2e}, eps cond(L) {EPS * cond:.2e}", flush=True)
    assert max(be) <= EPS * cond


@pytest.mark.parametrize("nbus,gamma,step", [(203, 1e6, 19), (500, 1e4, 19), (500, 1e6, 10)])
def test_late_interior_point_fronts(nbus, gamma, step):
    """H_gamma of late steps (Ds up to 1e8) and large gamma: no loss beyond the sums'
    own rounding, eps sqrt(n) of the norms."""
    g = GridPattern(nbus, int(1.3 * nbus), seed=11)
    sy = g.system(0, ds_range=ds_spread_schedule(step, 20))
    sy.gamma = gamma
    _, st, _, s = alone(g, sy)
    n, nz = st["n"], st["nnz_hgam"]
    rp, ci = s.debug(15, n + 1, np.int32), s.debug(16, nz, np.int32)
    v = s.debug(10, nz)
    rows = np.repeat(np.arange(n), np.diff(rp))
    a = np.zeros((n, n))
    low = ci <= rows
    a[rows[low], ci[low]] = v[low]
    a[ci[low], rows[low]] = v[low]
    be = backward_errors(a, a[rows, ci], rp, ci, np.random.default_rng(nbus))
    print(f"{nbus} {gamma:g} {step}: backward errors {max(be):.2e}", flush=True)
    assert max(be) <= EPS * np.sqrt(n)
