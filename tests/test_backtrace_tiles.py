"""The species backtrace at the edges of its 64 x 16 blocks, on small grids and for
displacements of more than a cell, against the numpy restatement."""
import numpy as np
import pytest

import passive_np as PN
import pmfmhd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-13), (np.float32, 2e-5)])
@pytest.mark.parametrize("n", [1, 2, 5, 17, 64, 65, 70])
@pytest.mark.parametrize("cells", [0.4, 3.0])
def test_backtrace_matches_numpy(n, cells, dtype, tol):
    """The sampled field varies by one per cell at most, so a position's rounding (2^-24 of n, three
    axes) bounds the difference: 2e-5 in float32, 1e-13 in float64."""
    rng = np.random.default_rng(n)
    U = np.zeros((9, n ** 3))
    U[0] = 1 + 0.2 * rng.random(n ** 3)
    U[1:4] = U[0] * rng.uniform(-1, 1, (3, n ** 3))
    U[4] = 3.0
    U = U.astype(dtype)
    s = M.allocate_state((n, n, n), 1.0 / n, dtype=dtype)
    s.set_conserved(U)
    a = [rng.random(n ** 3).astype(dtype) for _ in range(2)]
    dt = cells / n
    for mode in (2, 0, 1):
        b = [M.DeviceBuffer(n ** 3 * s.dtype.itemsize) for _ in range(4)]
        b[0].upload(a[0])
        b[1].upload(0.5 * a[1])
        if mode == 2:
            M.advect_passive_scalar(s, b[0], b[2], dt)
        elif mode == 0:
            M.advect_species(s, b[0], b[2], dt)
        else:
            M.advect_species(s, b[0], b[2], dt, species2=b[1], scratch2=b[3])
        got = b[0].download(dtype, n ** 3).astype(np.float64)
        U64 = U.astype(np.float64)
        if mode == 1:
            want, want2 = PN.backtrace(a[0].astype(float), U64, n, cells, mode=1, a2=0.5 * a[1].astype(float))
            got2 = b[1].download(dtype, n ** 3).astype(np.float64)
            assert np.abs(got2 - want2).max() <= tol
        else:
            want = PN.backtrace(a[0].astype(float), U64, n, cells, mode=mode)
        assert np.abs(got - want).max() <= tol, mode
