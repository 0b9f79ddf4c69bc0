"""The fold of a step's partial speeds beside the line between its two block sizes (2048 partials):
the speed it keeps is that of a fresh reduction, and a NaN anywhere stays one."""
import numpy as np
import pytest

import pmfmhd as M
from test_ref_dispatch import state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [12, 12 * 127, 12 * 128, 12 * 129])  # 16 workgroups for every twelve rows
def test_kept_speed_equals_a_fresh_reduction(ny):
    s = state((256, ny, 1), np.float64)
    M.step(s, 1e-3, ch=3.0, integrator="cube")
    kept = M.max_wavespeed(s)
    U = s.conserved()
    s.device_ptr(0)  # the next speed is a fresh reduction
    assert M.max_wavespeed(s) == kept
    for at in (0, U.shape[1] - 1):  # the first and the last workgroup's cells
        V = U.copy()
        V[1, at] = np.nan
        s.set_conserved(V)
        M.step(s, 1e-3, ch=3.0, integrator="cube")
        assert np.isnan(M.max_wavespeed(s))
