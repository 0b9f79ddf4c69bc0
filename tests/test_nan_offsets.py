"""A NaN cell: what a float64 PPM step makes of its neighbours' one-sided differences."""
import numpy as np
import pytest

import oracle as O
import pmfmhd as M
from test_gpu_parity import smooth_state

pytestmark = pytest.mark.gpu
DIMS = (18, 14, 9)


@pytest.mark.parametrize("integrator", ["cube", "ref"])
@pytest.mark.parametrize("per_cell", [False, True])
def test_nan_reaches_as_far_as_in_the_oracle(integrator, per_cell):
    """The reconstruction's offsets of a neighbour are NaN too, so the step's reach is two cells along
    each axis (glm_physics.jl:188-200)."""
    U = smooth_state(DIMS, seed=2).reshape(9, *DIMS[::-1])
    U[7, 4, 6, 8] = np.nan
    o = O.OracleState(DIMS, 0.1, dtype=np.float64, recon="ppm")
    s = M.allocate_state(DIMS, 0.1, dtype=np.float64, recon="ppm")
    M.set_ct_kernel(s, per_cell)
    for x in (o, s):
        x.set_conserved(U.reshape(9, -1))
    o.step(1e-3, ch=3.0)
    M.step(s, 1e-3, ch=3.0, integrator=integrator)
    want = np.isnan(np.asarray(o.U)).reshape(U.shape)[7]
    got = np.isnan(s.conserved()).reshape(U.shape)[7]
    for axis, at in enumerate((4, 6, 8)):
        for d in (-2, -1, 1, 2):
            c = [4, 6, 8]
            c[axis] = at + d
            assert want[tuple(c)] and got[tuple(c)], (axis, d)
