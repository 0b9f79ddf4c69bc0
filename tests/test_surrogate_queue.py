"""The network's batches of a plane's smooth faces: each face's result is its own, whatever
shares its batch, so a state repeated along y and z steps to its own repetition, bit for bit,
from planes with fewer faces than a batch to full queues."""
import os

import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P
from pmfmhd.surrogate import Surrogate, step_surrogate

pytestmark = pytest.mark.gpu
WEIGHTS = os.path.join(os.path.dirname(M.__file__), "data", "surrogate_weights.npy")


@pytest.mark.parametrize("dims", [(16, 2, 2), (16, 3, 5), (16, 5, 3)])
@pytest.mark.parametrize("rough", [0.0, 0.5, 0.97])
def test_repeated_state_steps_to_its_repetition(dims, rough):
    nx, ny, nz = dims
    n = nx * ny * nz
    rng = np.random.default_rng(int(100 * rough) + n)
    one = np.ones(n)
    bad = rng.random(n) < rough
    rho = one + 1e-3 * rng.normal(size=n) + np.where(bad, 0.5 * rng.random(n), 0)
    q = [rho, *(0.05 * rng.normal(size=(3, n))), one + 1e-3 * rng.normal(size=n),
         *(0.3 + 1e-3 * rng.normal(size=(3, n))), 0 * one]
    U = P.prim2cons(q, 5.0 / 3.0).astype(np.float32).reshape(9, nz, ny, nx)
    base = None
    for ry, rz in ((1, 1), (2, 1), (3, 4), (7, 2)):
        V = np.tile(U, (1, rz, ry, 1))
        s = M.allocate_state((nx, ny * ry, nz * rz), 0.1, dtype=np.float32, recon="plm_minmod")
        s.set_conserved(V.reshape(9, -1))
        net = Surrogate(s, seed=1)
        net.set_weights(np.load(WEIGHTS))
        count = step_surrogate(s, net, 0.004, 2.5, thr=0.02, count=True)
        got = s.conserved().reshape(V.shape)
        if base is None:
            base, faces = got, count
        assert count == faces * ry * rz
        assert np.array_equal(got, np.tile(base, (1, rz, ry, 1)))
