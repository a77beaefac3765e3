"""The factorization's second stream runs beside the solver's own: it is picked by a
test that tells streams on one hardware queue from streams on two.  Needs an MI355X."""
import numpy as np
import pytest

import hykkt_amd as H
from hykkt_amd.generator import GridPattern
from test_gpu_batch_engine import alone

pytestmark = pytest.mark.gpu


def test_picked_stream_overlaps():
    g = GridPattern(203, 263, seed=11, gamma=1e5)
    rc, _, _, s = alone(g, g.system(0))
    assert rc == H.HYKKT_OK
    picked, same = s.debug(23, 2, np.int32)
    assert picked == 1   # on an idle device, of at most four candidates
    assert same == 0     # a stream never runs beside itself
    assert s.execute() == H.HYKKT_OK   # the test left the stream as it was
