"""pmf_autotune's depth and time belong together, also on grids that keep a shorter built-in depth."""
import time

import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P

pytestmark = pytest.mark.gpu


def test_the_returned_depth_takes_the_returned_time():
    """At 16^3 the built-in choice (one plane) takes half of the time of four planes. The bound is
    wide enough for a queued step's launch, which the tuner's events leave out or not."""
    s = M.allocate_state((16, 16, 16), 1 / 16, dtype=np.float32, recon="plm_minmod")
    s.set_conserved(P.config_state("bstatic_32", seed=3, n=16))
    zc, ms = M.autotune(s, reps=200)
    M.set_chunk(s, zc)
    best = 1e9
    for _ in range(5):
        s.synchronize()
        t = time.perf_counter()
        for _ in range(200):
            M.step(s, 1e-6, ch=3.0, integrator="cube")
        s.synchronize()
        best = min(best, (time.perf_counter() - t) / 200 * 1e3)
    assert 0.75 * best <= ms <= 2 * best
