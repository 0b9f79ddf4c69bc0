"""A reflecting axis of one cell: the per-cell step's second ghost layer stays in the grid."""
import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 1, 6), (1, 4, 5), (6, 7, 1)])
def test_step_on_a_reflecting_axis_of_one_cell(dims):
    """At rest and uniform apart from a field along the thin axis's neighbours, every ghost cell equals
    the cell itself, so the state stays as it is; the fused step still refuses the grid."""
    n = int(np.prod(dims))
    one, zero = np.ones(n), np.zeros(n)
    bcs = tuple("reflecting" if d == 1 else "outflow" for d in dims)
    s = M.allocate_state(dims, 0.1, dtype=np.float64, bcs=bcs)
    U = P.prim2cons([one, zero, zero, zero, one, zero, zero, zero, zero], 5.0 / 3.0)
    s.set_conserved(U)
    M.step(s, 1e-3, ch=3.0)
    assert np.abs(s.conserved() - U).max() <= 1e-15
    with pytest.raises(M.MHDError, match="reflecting axes two"):
        M.step(s, 1e-3, ch=3.0, integrator="cube")
