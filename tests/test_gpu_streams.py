"""Several solvers alive in one process, more streams than the default number of
hardware queues: each one's look-ahead stream is picked on its own, and all
give the same bits.  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H
from hykkt_amd.generator import GridPattern
from test_gpu_batch_engine import alone

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 6])
def test_solvers_sharing_queues(count):
    g = GridPattern(700, 910, seed=3, gamma=1e5)
    sy = g.system(0)
    runs = [alone(g, sy) for _ in range(count)]   # all kept alive
    assert all(r[0] == H.HYKKT_OK for r in runs)
    for r in runs[1:]:
        assert np.array_equal(r[2], runs[0][2])
    for _, _, x, s in runs:                       # and again, in turn
        assert s.execute() == H.HYKKT_OK
        assert np.array_equal(np.concatenate(s.solution()), x)
    assert runs[0][1]["resid4"] <= 1e-8
