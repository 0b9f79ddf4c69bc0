"""The masked fallback in the instances that load a pass ahead (its flags are among the values
loaded early): a state repeated along every axis steps to its own repetition, bit for bit."""
import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(48, 48, 40), (50, 41, 42)])
@pytest.mark.parametrize("recon,riemann", [("plm_minmod", "hlld"), ("plm", "hll")])
@pytest.mark.parametrize("share", [0.05, 1.0])
def test_flagged_state_steps_to_its_repetition(dims, recon, riemann, share):
    nx, ny, nz = dims
    n = nx * ny * nz
    rng = np.random.default_rng(9)
    one = np.ones(n)
    q = [one + 0.2 * rng.uniform(-1, 1, n), *rng.normal(0, 0.3, (3, n)), one, *rng.normal(0, 0.4, (3, n)),
         rng.normal(0, 0.05, n)]
    U = P.prim2cons(q, 5.0 / 3.0).astype(np.float32).reshape(9, nz, ny, nx)
    corr = np.zeros((9, nz, ny, nx))
    corr[1:4] = 0.01 * rng.normal(size=(3, nz, ny, nx))
    corr[4] = rng.random((nz, ny, nx)) < share
    out = []
    for r, masked in ((1, True), (2, True), (1, False)):  # 960 workgroups of four planes; an eighth of them
        s = M.allocate_state((r * nx, r * ny, r * nz), 0.1, dtype=np.float32, recon=recon, riemann=riemann)
        s.set_conserved(np.tile(U, (1, r, r, r)).reshape(9, -1))
        M.set_chunk(s, 4)
        buf = M.correction_buffer(s, np.tile(corr, (1, r, r, r)).reshape(9, -1))
        M.load_psi(s, buf)
        M.step_radiation(s, 2e-3, 3.0, 0.98, 0.2, buf, track_density=False, fallback=masked, integrator="cube")
        out.append(s.conserved().reshape(9, r * nz, r * ny, r * nx))
    assert np.all(np.isfinite(out[0]))
    assert np.array_equal(np.tile(out[0], (1, 2, 2, 2)), out[1])
    assert not np.array_equal(out[0], out[2])  # the flags act
