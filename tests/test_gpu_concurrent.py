"""Solvers of several threads busy on the device at once: the waves of a workgroup then
share their SIMDs with other solvers' work and drift apart, and every execute has to
give the bits it gives alone.  Needs an MI355X."""
import threading
import time

import numpy as np
import pytest

import hykkt_amd as H
from hykkt_amd.generator import GridPattern
from test_gpu_batch_engine import batched, draws

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbus,count,threads", [(1_000, 16, 8), (5_000, 4, 4)])
def test_concurrent_solvers_same_bits(nbus, count, threads):
    g = GridPattern(nbus, int(1.3 * nbus), seed=11, gamma=1e5)
    systems = draws(g, count, [(1e-2, 1e2), (1e-4, 1e6)], [1e5])
    solvers = []
    for _ in range(threads):
        b, rc = batched(g, systems, device=True, sweep_share=4)
        assert rc == [H.HYKKT_OK] * count
        solvers.append(b)
    ref = [np.concatenate(solvers[0].solution_k(k)) for k in range(count)]
    keys = ("pivot", "cg_iters", "refine_steps", "resid2", "resid4")
    want = [[solvers[0].stats_k(k)[key] for key in keys] for k in range(count)]
    end = time.perf_counter() + 3.0
    bad, runs = [], [0] * threads

    def work(i):
        while time.perf_counter() < end and not bad:
            rc = solvers[i].execute_batch(count)
            got = [[solvers[i].stats_k(k)[key] for key in keys] for k in range(count)]
            if rc != [H.HYKKT_OK] * count or got != want:
                bad.append((i, runs[i], rc, got))
            runs[i] += 1

    pool = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    print("executes", runs, flush=True)
    assert not bad, bad[0]
    for b in solvers:
        for k in range(count):
            assert np.array_equal(np.concatenate(b.solution_k(k)), ref[k])
