"""Refinement passes whose CG outlasts the host's first look at it: the solution must
not depend on when the host looks (cg_check_every, the iterations of the calls
before) or on the other systems of a batch.  Small gammas and wide Ds spreads, so the
corrections' CG takes several iterations.  Needs an MI355X."""
import numpy as np
import pytest

import _oracle as O
import hykkt_amd as H
from hykkt_amd.generator import GridPattern
from test_gpu_batch_engine import alone, batched

pytestmark = pytest.mark.gpu

KEYS = ("cg_iters", "cg_status", "refine_steps", "resid2", "resid4", "resid4_first")


def same(st, x, ref):
    assert np.array_equal(x, ref[2])
    for key in KEYS:
        assert st[key] == ref[1][key], key


@pytest.mark.parametrize("seed", [0, 1])
@pytest.mark.parametrize("gamma", [1e1, 1e2, 1e3])
def test_looks_do_not_change_the_solution(gamma, seed):
    g = GridPattern(203, 263, seed=11)
    sy = g.system(seed, ds_range=(1e-4, 1e8))
    sy.gamma = gamma
    opts = dict(refine_tol=1e-13)
    # one look, after the iteration limit: recovery and residual run once a pass
    ref = alone(g, sy, cg_check_every=100, **opts)
    print(gamma, seed, {k: ref[1][k] for k in KEYS}, flush=True)
    assert ref[0] == H.HYKKT_OK and ref[1]["refine_steps"] >= 1
    for every in (0, 1, 2):
        rc, st, x, s = alone(g, sy, cg_check_every=every, **opts)
        same(st, x, ref)
        assert s.execute() == H.HYKKT_OK   # with the hints the first call left
        same(s.stats(), np.concatenate(s.solution()), ref)
    c = lambda m: O.Csr(m.n, m.m, m.rp, m.ci, m.v)
    orc = O.execute(c(sy.H), sy.Ds.v, c(sy.Jc), c(sy.Jd), sy.rx, sy.rs, sy.ry, sy.ryd, gamma,
                    perm=ref[3].permutation())
    # the default options stop refining at 9e-9; the 1e-8 target and the oracle agree
    rc, st, x, _ = alone(g, sy)
    xo = np.concatenate([orc["dx"], orc["ds"], orc["dyc"], orc["dyd"]])
    assert st["resid4"] <= 1e-8
    assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)


@pytest.mark.parametrize("every", [0, 1])
def test_batch_of_unequal_iterations(every):
    """Systems that stop beside one whose corrections go on iterating."""
    g = GridPattern(203, 263, seed=11)
    systems = []
    for k, gamma in enumerate((1e6, 1e1, 1e4, 1e2)):
        sy = g.system(k, ds_range=(1e-4, 1e8))
        sy.gamma = gamma
        systems.append(sy)
    opts = dict(refine_tol=1e-13)
    b, rc = batched(g, systems, cg_check_every=every, **opts)
    for _ in range(2):   # and again, with the hints the first call left
        for k, sy in enumerate(systems):
            ref = alone(g, sy, cg_check_every=100, **opts)
            assert rc[k] == ref[0] == H.HYKKT_OK
            same(b.stats_k(k), np.concatenate(b.solution_k(k)), ref)
        rc = b.execute_batch(len(systems))


@pytest.mark.parametrize("every", [0, 1])
def test_early_looks_run_no_recovery(every):
    """Looks at a CG that is not done read its live flags alone: at most two recoveries
    and residuals a pass (k_spmv in the profile has both, and the products)."""
    g = GridPattern(203, 263, seed=11)
    sy = g.system(0, ds_range=(1e-4, 1e8))
    sy.gamma = 1e1
    opts = dict(refine_max=0, cg_check_every=every)
    _, st, _, s = alone(g, sy, **opts)
    assert st["cg_iters"] > 10
    for _ in range(2):
        s.profile(True)
        s.execute()
        n = s.kernel_times()["k_spmv"]["launches"]
        # Jd^T, Jc^T and Jc once, and both Jc products per iteration
        assert 2 <= n - (3 + 2 * s.stats()["cg_iters"]) <= 4
        s.profile(False)
    # a fresh pattern, whose iteration count is not known
    s = H.HykktSolver(sy.gamma)
    s.options(**opts)
    s.profile(True)
    d = g.d
    s.set_H(sy.H.rp, sy.H.ci, sy.H.v, g.n, g.n, g.H.nnz)
    s.set_Ds(np.arange(d + 1), np.arange(d), sy.Ds.v, d, d, d)
    s.set_Jc(sy.Jc.rp, sy.Jc.ci, sy.Jc.v, g.m, g.n, g.Jc.nnz)
    s.set_Jd(sy.Jd.rp, sy.Jd.ci, sy.Jd.v, g.d, g.n, g.Jd.nnz)
    for name in ("rx", "rs", "ry", "ryd"):
        v = getattr(sy, name)
        getattr(s, "set_" + name)(v, len(v))
    s.execute()
    assert s.kernel_times()["k_spmv"]["launches"] == 3 + 2 * s.stats()["cg_iters"] + 2
