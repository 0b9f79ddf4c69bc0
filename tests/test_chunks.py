"""The built-in z-chunk choice: the state after a step has the same bits whatever the chunk."""
import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(16, 12, 1), (17, 13, 5), (32, 32, 32), (40, 25, 83)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("solver,recon", [("glm", "plm_minmod"), ("glm", "ppm"), ("ct", "plm")])
def test_step_does_not_depend_on_the_chunk(dims, dtype, solver, recon):
    rng = np.random.default_rng(2)
    n = int(np.prod(dims))
    one = np.ones(n)
    q = [one + 0.1 * rng.uniform(-1, 1, n), *rng.normal(0, 0.3, (3, n)), one, *rng.normal(0, 0.5, (3, n)), 0 * one]
    U = P.prim2cons(q, 5.0 / 3.0)
    out = []
    for zc in (0, 4, 7, 32):
        s = M.allocate_state(dims, 0.1, dtype=dtype, recon=recon, mhd_solver=solver)
        s.set_conserved(U)
        if solver == "ct":
            M.ct_install_faces(s, *U[5:8])
        M.set_chunk(s, zc)
        dt, smax = M.compute_dt(s, 0.2)
        for _ in range(2):
            M.step(s, float(dt), ch=float(smax), integrator="ref" if solver == "ct" else "cube")
        out.append((s.conserved(), M.max_wavespeed(s)) + (tuple(s.ct_slot(d) for d in range(3)) if solver == "ct" else ()))
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
