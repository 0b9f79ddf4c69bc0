"""PPM CT steps that were told nothing about the workspace write slots 3-14, with the values of the
step that fills them for the separate edge pass (integrator_ref.jl:83-139)."""
import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(33, 13, 17), (16, 12, 5), (8, 5, 3), (48, 40, 30)])
@pytest.mark.parametrize("riemann", ["hlld", "hll", "llf"])
@pytest.mark.parametrize("wide", ["0", "1"])
def test_default_ppm_step_fills_the_workspace(dims, riemann, wide, monkeypatch):
    monkeypatch.setenv("PMFMHD_WIDE_OFFSETS", wide)
    n = int(np.prod(dims))
    rng = np.random.default_rng(11)
    one = np.ones(n)
    q = [one + 0.2 * rng.random(n), *rng.normal(0, 0.4, (3, n)), one, *rng.normal(0, 0.6, (3, n)), 0 * one]
    U = P.prim2cons(q, 5.0 / 3.0).astype(np.float32)
    out = []
    for fill in (True, None):
        s = M.allocate_state(dims, 1.0 / dims[0], dtype=np.float32, recon="ppm", riemann=riemann, mhd_solver="ct")
        if fill:
            M.set_ct_workspace(s, True)
        s.set_conserved(U)
        M.ct_faces_from_cells(s)
        for _ in range(3):
            dt, _ = M.compute_dt(s, 0.3)
            M.step(s, float(dt))
        out.append((s.conserved(), [s.ct_slot(k) for k in range(21)]))
    assert np.all(np.isfinite(out[1][0]))
    assert np.array_equal(out[0][0], out[1][0])
    for k in range(21):
        assert np.array_equal(out[0][1][k], out[1][1][k]), k
        assert k > 14 or np.any(out[1][1][k]), k
