"""Which kernel a :ref step takes on thin grids, where most of a fused workgroup's 16 x 12 columns
are empty: never much slower than the per-cell kernel, and the same bits."""
import time

import numpy as np
import pytest

import pmfmhd as M
from test_ref_dispatch import state

pytestmark = pytest.mark.gpu


def times(a, b, reps=50):
    """Time of a queued step of either state, the two timed in turn, the best of five."""
    best = [1e9, 1e9]
    for _ in range(5):
        for k, s in enumerate((a, b)):
            M.step(s, 1e-5, ch=3.0)
            s.synchronize()
            t = time.perf_counter()
            for _ in range(reps):
                M.step(s, 1e-5, ch=3.0)
            s.synchronize()
            best[k] = min(best[k], time.perf_counter() - t)
    return best


@pytest.mark.parametrize("dims", [(65536, 1, 1), (1, 1, 65536), (4, 4, 4096), (1, 256, 256), (256, 1, 256),
                                  (256, 256, 1), (32, 32, 32)])
@pytest.mark.parametrize("dtype,recon", [(np.float32, "plm"), (np.float64, "plm"), (np.float64, "ppm")])
def test_thin_grids_step_as_fast_as_the_per_cell_kernel(dims, dtype, recon):
    """A third is more than the choice's model errs by; the fused kernel takes 1.4 to 40 times the
    per-cell kernel's time on the thinnest of these grids and half of it on the cube."""
    a, b = (state(dims, dtype, recon=recon) for _ in range(2))
    M.set_ct_kernel(b, True)
    if recon == "plm":
        M.step(a, 1e-4, ch=3.0)
        M.step(b, 1e-4, ch=3.0)
        assert np.array_equal(a.conserved(), b.conserved())
    chosen, per_cell = times(a, b)
    assert chosen <= 1.33 * per_cell
    if dims == (32, 32, 32):
        assert chosen <= 0.8 * per_cell
