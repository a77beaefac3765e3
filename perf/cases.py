"""The solver's performance cases: what a program using this framework has it do,
from single small KKT systems to 40,000-bus ones, alone, in same-pattern
sequences and in batches, and the component entry points.

Every case names a grid (buses, branches), the penalty gamma and the place in an
interior-point run (`step` of 20: the spread of Ds grows from 1e-2..1e2 to
1e-4..1e8; -1: Ds log-uniform on 1e-4..1e4, the single-system workloads).  The
sparsity pattern is fixed by the sizes; the values come from the seed.

kind "solve": HykktSolver on a pattern it has analysed (the same-pattern
sequence of an interior-point method): bind the next system's values, execute,
read the solution back.  device: values resident in HBM (inputs_on_device)
instead of host arrays.
kind "batch": BatchSolver, `count` systems of one pattern in one call.
kind "component": the Cholesky and Schur-CG entry points on host arrays:
factor, solve, conjugate gradient on J A^{-1} J^T.
"""
from __future__ import annotations

import functools
import math

import numpy as np

import hykkt_amd as H
from hykkt_amd.generator import GridPattern, ds_spread_schedule

# Grid sizes from the benchmark's workloads: single systems of 500 to 80,000
# buses, served patterns of 1,000, 5,000 and 20,000 buses, batches of 200 to
# 5,000.  40,000 is the largest here (80,000 takes 5 s a solve).
PLAIN_RANGE = (200, 40_000)
BATCH_RANGE = (200, 5_000)
BRANCHES = 1.3


def listed():
    return [
        # the smallest call: a small grid through the drop-in path, host arrays;
        # latency and launches are all there is
        _solve("solve 203 host", 203, 1e4, -1, device=False),
        # the 500-bus / 700-branch single system, as a drop-in caller binds it
        _solve("solve 500 host", 500, 1e4, -1, device=False, nbranch=700),
        # one served pattern of each size, a request at a time, values in HBM
        _solve("solve 1000 device", 1_000, 1e5, 4, device=True),
        _solve("solve 5000 device", 5_000, 1e5, 7, device=True),
        # the 10,000-bus / 13,000-branch sequence, an early step; and one near
        # its end (refinement passes) from host arrays
        _solve("solve 10000 device", 10_000, 1e5, 2, device=True, nbranch=13_000),
        _solve("solve 10000 host late", 10_000, 1e5, 18, device=False, nbranch=13_000),
        _solve("solve 20000 device", 20_000, 1e5, 5, device=True),
        # the large single system: factorization-bound
        _solve("solve 40000 device", 40_000, 1e6, 0, device=True, nbranch=55_000),
        # a served slot's full batch of 1,000-bus requests
        _batch("batch 16 x 1000", 16, 1_000, 1e5, 3, device=True),
        # an odd-sized pattern of the 256-system batch: eight draws, host arrays
        _batch("batch 8 x 2477 host", 8, 2_477, 1e5, -1, device=False),
        # a served slot's full batch of 5,000-bus requests
        _batch("batch 8 x 5000", 8, 5_000, 1e5, 6, device=True),
        # the component classes: factor, solve and Schur CG at a 1,000-bus grid's size
        dict(name="component 1000", kind="component", nbus=1_000, nbranch=1_300),
    ]


def _solve(name, nbus, gamma, step, device, nbranch=None):
    return dict(name=name, kind="solve", nbus=nbus, nbranch=nbranch or int(BRANCHES * nbus),
                gamma=gamma, step=step, device=device)


def _batch(name, count, nbus, gamma, step, device):
    return dict(_solve(name, nbus, gamma, step, device), kind="batch", count=count)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "batch", "batch", "component"])
    if kind == "component":
        nbus = _log_int(rng, 200, 3_000)
        return dict(kind=kind, nbus=nbus, nbranch=int(nbus * rng.uniform(1.2, 1.4)))
    lo, hi = PLAIN_RANGE if kind == "solve" else BATCH_RANGE
    nbus = _log_int(rng, lo, hi)
    c = dict(kind=kind, nbus=nbus, nbranch=int(nbus * rng.uniform(1.25, BRANCHES + 0.02)),
             gamma=10.0 ** rng.uniform(4.0, 6.0), step=rng.randrange(-1, 20),
             device=rng.random() < 0.6)
    if kind == "batch":
        c["count"] = rng.randint(2, 16 if nbus <= 2_000 else 8)
    return c


# ---------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=4)
def _grid(nbus, nbranch):
    return GridPattern(nbus, nbranch, seed=11)


def _ds_range(case):
    return (1e-4, 1e4) if case["step"] < 0 else ds_spread_schedule(case["step"], 20)


def _systems(case, seed):
    g = _grid(case["nbus"], case["nbranch"])
    count = case.get("count", 1)
    return [g.system(seed * 64 + k, ds_range=_ds_range(case)) for k in range(count)]


def _values(sy):
    return [sy.H.v, sy.Ds.v, sy.Jc.v, sy.Jd.v, sy.rx, sy.rs, sy.ry, sy.ryd]


class _Pattern:
    """The grid's index arrays, on the host or in HBM, bound to a solver with one
    system's values."""

    def __init__(self, g, device):
        d = g.d
        put = H.DeviceArray if device else (lambda a: a)
        i32 = lambda a: put(np.ascontiguousarray(a, dtype=np.int32))
        self.g, self.put = g, put
        self.idx = [(i32(g.H.rp), i32(g.H.ci)), (i32(np.arange(d + 1)), i32(np.arange(d))),
                    (i32(g.Jc.rp), i32(g.Jc.ci)), (i32(g.Jd.rp), i32(g.Jd.ci))]

    def bind(self, s, v):
        g, (h, ds, jc, jd) = self.g, self.idx
        s.set_H(*h, v[0], g.n, g.n, g.H.nnz)
        s.set_Ds(*ds, v[1], g.d, g.d, g.d)
        s.set_Jc(*jc, v[2], g.m, g.n, g.Jc.nnz)
        s.set_Jd(*jd, v[3], g.d, g.n, g.Jd.nnz)
        s.set_rx(v[4], g.n)
        s.set_rs(v[5], g.d)
        s.set_ry(v[6], g.m)
        s.set_ryd(v[7], g.d)


def prepare(case, seed):
    if case["kind"] == "component":
        return _prepare_component(case, seed)
    g = _grid(case["nbus"], case["nbranch"])
    p = _Pattern(g, case["device"])
    vals = [[p.put(a) for a in _values(sy)] for sy in _systems(case, seed)]
    # the plan such a program keeps: the analysis (and the launch shapes chosen
    # for it) of a first execute on the pattern's base values
    first = [p.put(a) for a in _values(g.system(-1, ds_range=_ds_range(case)))]
    if case["kind"] == "solve":
        s = H.HykktSolver(case["gamma"])
        if case["device"]:
            s.options(inputs_on_device=1)
        p.bind(s, first)
        s.execute()
    else:
        s = H.BatchSolver(case["gamma"], case["count"])
        if case["device"]:
            s.options(inputs_on_device=1)
        p.bind(s, first)
        for k in range(case["count"]):
            s.bind_system(k, case["gamma"], *first)
        s.execute_batch(case["count"])
    return dict(kind=case["kind"], s=s, p=p, vals=vals, gamma=case.get("gamma"), first=first)


def run(state):
    s = state["s"]
    if state["kind"] == "component":
        fail = s.factor(state["a"])
        x = s.solve(state["b"])
        y, status, _, _ = s.schur_cg(*state["j"], state["r"])
        return dict(fail=fail, x=x, status=status, y=y)
    if state["kind"] == "solve":
        state["p"].bind(s, state["vals"][0])
        status = s.execute()
        dx, ds, dyc, dyd = s.solution()
        return dict(status=status, dx=dx, ds=ds, dyc=dyc, dyd=dyd)
    vals = state["vals"]
    for k, v in enumerate(vals):
        s.bind_system(k, state["gamma"], *v)
    status = s.execute_batch(len(vals))
    sol = [s.solution_k(k) for k in range(len(vals))]
    return dict(status=status, **{n: np.stack([x[i] for x in sol])
                                  for i, n in enumerate(("dx", "ds", "dyc", "dyd"))})


# ---------------------------------------------------------------- components
COMPONENT_GAMMA = 1e4


@functools.lru_cache(maxsize=4)
def _neighbour_pairs(nbus, nbranch):
    """Pairs of buses with a common closed neighbour: (first, second, and their places
    among the 4-entry groups of Jc's bus rows, which list a bus's closed
    neighbourhood in order)."""
    e = _grid(nbus, nbranch).edges
    own = np.arange(nbus)
    a = np.concatenate([own, e[:, 0], e[:, 1]])    # row bus -> closed neighbourhood
    b = np.concatenate([own, e[:, 1], e[:, 0]])
    order = np.lexsort((b, a))
    a, b = a[order], b[order]
    ptr = np.searchsorted(a, np.arange(nbus + 1))
    deg = np.diff(ptr)
    left = np.repeat(np.arange(len(a)), deg[a])
    off = np.arange(len(left)) - np.repeat(np.cumsum(deg[a]) - deg[a], deg[a])
    right = np.repeat(ptr[a], deg[a]) + off
    return b[left], b[right], left, right, a, ptr


@functools.lru_cache(maxsize=4)
def _hgamma_pattern(nbus, nbranch):
    """CSR pattern of H + Jd^T Jd + Jc^T Jc: buses couple where some bus is next
    to (or is) both.  Also each entry's row."""
    p, q = _neighbour_pairs(nbus, nbranch)[:2]
    key = np.unique(p.astype(np.int64) * nbus + q)
    r, c = key // nbus, key % nbus
    blk = np.arange(4)
    rows = (4 * r[:, None, None] + blk[None, :, None]).repeat(4, axis=2).ravel()
    cols = (4 * c[:, None, None] + blk[None, None, :]).repeat(4, axis=1).ravel()
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    rp = np.searchsorted(rows, np.arange(4 * nbus + 1)).astype(np.int32)
    return rp, cols.astype(np.int32), rows.astype(np.int32)


@functools.lru_cache(maxsize=4)
def _ordered_pattern(nbus, nbranch):
    """That pattern in the fill-reducing order a caller factorizes it in, each
    entry's row, and the inverse of the order."""
    rp, ci, rows = _hgamma_pattern(nbus, nbranch)
    perm = H.amd_order(rp, ci)
    inv = np.empty(len(perm), np.int64)
    inv[perm] = np.arange(len(perm))
    r, c = inv[rows], inv[ci]
    order = np.lexsort((c, r))
    r, c = r[order], c[order]
    rp = np.searchsorted(r, np.arange(len(perm) + 1)).astype(np.int32)
    return rp, c.astype(np.int32), r, inv


def _component_inputs(case, seed):
    """A = D + gamma J^T J in its fill-reducing order (D diagonally dominant on the
    same pattern), J in that order of its columns, and right-hand sides."""
    size = case["nbus"], case["nbranch"]
    rng = np.random.default_rng([seed, 17])
    g = _grid(*size)
    rp, ci, r, inv = _ordered_pattern(*size)
    n = len(rp) - 1
    lower = r >= ci
    v = np.zeros(len(ci))
    v[lower] = rng.standard_normal(int(lower.sum()))
    # the mirror of (r, c) is (c, r): sorting by (c, r) lists the mirrors in order
    mirror = np.lexsort((r, ci))
    v = np.where(lower, v, v[mirror])
    v[r == ci] = np.bincount(r, np.abs(v), minlength=n) + rng.uniform(0.5, 2.0, n)
    jv = g.Jc.v * (1.0 + 0.05 * rng.standard_normal(g.Jc.nnz))
    # + gamma J^T J, the 4 x 4 blocks of every pair of a bus row's neighbours
    p, q, left, right, a, ptr = _neighbour_pairs(*size)
    at = [g.Jc.rp[2 * a + k] + 4 * (np.arange(len(a)) - ptr[a]) for k in (0, 1)]
    rows = [jv[x[:, None] + np.arange(4)[None, :]] for x in at]
    blocks = sum(w[left][:, :, None] * w[right][:, None, :] for w in rows)
    br = inv[(4 * p[:, None, None] + np.arange(4)[None, :, None]).repeat(4, axis=2)]
    bc = inv[(4 * q[:, None, None] + np.arange(4)[None, None, :]).repeat(4, axis=1)]
    pos = np.searchsorted(r * n + ci, (br * n + bc).ravel())
    v += COMPONENT_GAMMA * np.bincount(pos, blocks.ravel(), minlength=len(v))
    v = np.where(lower, v, v[mirror])
    # J's columns in the same order
    jr = np.repeat(np.arange(g.m), np.diff(g.Jc.rp))
    jc = inv[g.Jc.ci]
    order = np.lexsort((jc, jr))
    j = (g.Jc.rp, jc[order].astype(np.int32), jv[order])
    return (rp, ci, r, v), j, rng.standard_normal(n), rng.standard_normal(g.m)


def _prepare_component(case, seed):
    (rp, ci, _, v), j, b, r = _component_inputs(case, seed)
    s = H.Cholesky(rp, ci)
    s.factor(v)
    return dict(kind="component", s=s, a=v, b=b, j=j, r=r)


# ---------------------------------------------------------------- work
@functools.lru_cache(maxsize=64)
def _factor_work(nbus, nbranch):
    rp, ci = _ordered_pattern(nbus, nbranch)[:2]
    a = H.chol_analyze_host(rp, ci)
    return a["flops"], a["nnz_l"]


def work(case):
    """Inputs read once, the solution written once; the factorization's flops, and
    one triangular-solve pair for each of the right-hand side and the first
    product of the conjugate gradient."""
    g = _grid(case["nbus"], case["nbranch"])
    flops, nnz_l = _factor_work(case["nbus"], case["nbranch"])
    count = case.get("count", 1)
    if case["kind"] == "component":
        nnz = len(_ordered_pattern(case["nbus"], case["nbranch"])[1])
        nbytes = 8.0 * (nnz + g.Jc.nnz + 2 * (g.n + g.m))
    else:
        nbytes = 8.0 * (g.H.nnz + g.Jc.nnz + g.Jd.nnz + g.d + 2 * (g.n + g.m + 2 * g.d))
    return {"bytes": count * nbytes, "flops": count * (flops + 8.0 * nnz_l)}


# ---------------------------------------------------------------- exact
EXACT_MOST = 4.0   # dense solves, in units of a 1,000-bus system's, that take seconds


def _csr_mul(rp, ci, v, x):
    t = v * x[ci]
    out = np.zeros(len(rp) - 1, t.dtype)
    full = np.diff(rp) > 0
    if len(t):
        out[full] = np.add.reduceat(t, rp[:-1][full])
    return out


def _csr_tmul(rp, ci, v, x, ncol):
    t = v * np.repeat(x, np.diff(rp))
    order = np.argsort(ci, kind="stable")
    c = ci[order]
    out = np.zeros(ncol, t.dtype)
    if len(t):
        first = np.flatnonzero(np.concatenate([[True], c[1:] != c[:-1]]))
        out[c[first]] = np.add.reduceat(t[order], first)
    return out


def _dense(rp, ci, v, ncol):
    a = np.zeros((len(rp) - 1, ncol))
    a[np.repeat(np.arange(len(rp) - 1), np.diff(rp)), ci] = v
    return a


def _exact_kkt(sy):
    """The KKT system's solution: dense inverse of the system reduced to (dx, dyc),
    refined on the four block rows with extended-precision residuals."""
    n, m = len(sy.rx), len(sy.ry)
    ld = np.longdouble
    ds = sy.Ds.v
    jd, jc = _dense(sy.Jd.rp, sy.Jd.ci, sy.Jd.v, n), _dense(sy.Jc.rp, sy.Jc.ci, sy.Jc.v, n)
    k = np.zeros((n + m, n + m))
    k[:n, :n] = _dense(sy.H.rp, sy.H.ci, sy.H.v, n) + jd.T @ (ds[:, None] * jd)
    if not _definite(k[:n, :n] + 1e6 * (jc.T @ jc)):
        return None
    k[:n, n:], k[n:, :n] = jc.T, jc
    inv = np.linalg.inv(k)
    hv, jcv, jdv, dsl = (a.astype(ld) for a in (sy.H.v, sy.Jc.v, sy.Jd.v, ds))
    rhs = [a.astype(ld) for a in (sy.rx, sy.rs, sy.ry, sy.ryd)]
    dx, dsv, dy, dyd = (np.zeros_like(rhs[0]), np.zeros_like(rhs[1]), np.zeros_like(rhs[2]),
                        np.zeros_like(rhs[3]))
    for _ in range(5):
        ex = rhs[0] - (_csr_mul(sy.H.rp, sy.H.ci, hv, dx) + _csr_tmul(sy.Jc.rp, sy.Jc.ci, jcv, dy, n)
                       + _csr_tmul(sy.Jd.rp, sy.Jd.ci, jdv, dyd, n))
        es = rhs[1] - (dsl * dsv - dyd)
        ey = rhs[2] - _csr_mul(sy.Jc.rp, sy.Jc.ci, jcv, dx)
        ed = rhs[3] - (_csr_mul(sy.Jd.rp, sy.Jd.ci, jdv, dx) - dsv)
        t = ex + _csr_tmul(sy.Jd.rp, sy.Jd.ci, jdv, dsl * ed + es, n)
        z = inv @ np.concatenate([t, ey]).astype(np.float64)
        cx, cy = z[:n].astype(ld), z[n:].astype(ld)
        cs = _csr_mul(sy.Jd.rp, sy.Jd.ci, jdv, cx) - ed
        dx, dsv, dy, dyd = dx + cx, dsv + cs, dy + cy, dyd + (dsl * cs - es)
    return [np.asarray(a, dtype=np.float64) for a in (dx, dsv, dy, dyd)]


def _definite(a):
    try:
        np.linalg.cholesky(a)
        return True
    except np.linalg.LinAlgError:
        return False


def exact(case, seed):
    if case.get("count", 1) * (case["nbus"] / 1_000) ** 3 > EXACT_MOST:
        return None
    if case["kind"] == "component":
        (rp, ci, r, v), j, b, rhs = _component_inputs(case, seed)
        n = len(b)
        a = np.zeros((n, n))
        a[r, ci] = v
        x = np.linalg.solve(a, b)
        x = x + np.linalg.solve(a, (b.astype(np.longdouble) - _csr_mul(
            rp, ci, v.astype(np.longdouble), x)).astype(np.float64))
        jd = _dense(*j, n)
        y = np.linalg.solve(jd @ np.linalg.solve(a, jd.T), rhs)
        return dict(fail=None, x=x, status=None, y=y)
    sol = [_exact_kkt(sy) for sy in _systems(case, seed)]
    if any(x is None for x in sol):
        return None
    names = ("dx", "ds", "dyc", "dyd")
    if case["kind"] == "solve":
        return dict(status=None, **dict(zip(names, sol[0])))
    return dict(status=None, **{k: np.stack([x[i] for x in sol]) for i, k in enumerate(names)})
