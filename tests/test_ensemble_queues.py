"""The ensemble's work queues at their edges: fewer items than workgroups, one workgroup per
queue, queues of one item and empty ones."""
import numpy as np
import pytest

from pmfmhd import problems as P
from pmfmhd.ensemble import Ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edges", [[16], [16, 32], [48, 16, 16, 32]])
def test_queue_shapes_give_the_same_bits(edges):
    U = [P.random_mhd(n, seed=k + 1, kmax=n // 4) for k, n in enumerate(edges)]
    want = None
    for zc, nwg in ((None, None), (16, 8), (1, 8), (1, 1024), (5, 64), (16, 768)):
        e = Ensemble(edges)
        if nwg:
            e.set_config([min(zc, n) for n in edges], nwg)
        for c, u in enumerate(U):
            e.upload(c, u)
        e.run(3)
        e.run(2, graph=False)
        got = [e.download(c) for c in range(len(edges))] + list(e.clock())
        if want is None:
            want = got
        assert all(np.array_equal(a, b) for a, b in zip(want, got)), (zc, nwg)
