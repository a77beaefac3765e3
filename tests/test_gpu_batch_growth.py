"""A batch whose count changes from call to call, values and solutions in HBM: the
factor storage that an execute zeroes ahead for the next one, on the solver's second
stream, must be zero before a larger batch assembles into it.  Needs an MI355X."""
import threading

import numpy as np
import pytest

import hykkt_amd as H
from hykkt_amd.generator import GridPattern
from test_gpu_batch_engine import alone, batched, draws

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbus,busy", [(203, False), (5_000, False), (5_000, True)])
def test_growing_batch(nbus, busy):
    g = GridPattern(nbus, int(1.3 * nbus), seed=11, gamma=1e5)
    systems = draws(g, 8, [(1e-3, 1e4)], [1e5])
    b, rc = batched(g, systems, device=True)
    assert rc == [H.HYKKT_OK] * 8
    ref = [np.concatenate(b.solution_k(k)) for k in range(8)]
    assert np.array_equal(alone(g, systems[0])[2], ref[0])
    done = threading.Event()
    errors = []

    def other():
        # another solver's work, which delays this one's second stream
        try:
            o, _ = batched(g, systems[:2], device=True)
            while not done.is_set():
                assert o.execute_batch(2) == [H.HYKKT_OK] * 2
        except Exception as e:   # reported by the test's own thread
            errors.append(e)

    t = threading.Thread(target=other)
    if busy:
        t.start()
    try:
        # nothing read back in between: a copy on the null stream would wait for the
        # second stream
        for count in (1, 8, 2, 8, 1, 3, 8, 7, 8):
            assert b.execute_batch(count) == [H.HYKKT_OK] * count, count
            assert all(b.stats_k(k)["pivot"] < 0 for k in range(count)), count
    finally:
        done.set()
        if busy:
            t.join()
    assert not errors
    for k in range(8):
        assert np.array_equal(np.concatenate(b.solution_k(k)), ref[k]), k
