"""A reflecting axis of one cell: both ghost layers mirror the cell itself (the second one's mirror
image lies outside and is clamped), in a state whose slopes depend on both."""
import numpy as np
import pytest

import oracle as O
import pmfmhd as M
from pmfmhd import problems as P

DT, CH = 4e-3, 3.0


def conserved(dims):
    n = int(np.prod(dims))
    rng = np.random.default_rng(3)
    one = np.ones(n)
    # flow and field through the thin axis, larger than their variation: a mirrored cell is a large jump
    q = [one + 0.3 * rng.random(n), *(0.4 + 0.3 * rng.random((3, n))), one + 0.3 * rng.random(n),
         *(0.5 + 0.3 * rng.random((3, n))), 0.1 * rng.random(n)]
    return P.prim2cons(q, 5.0 / 3.0).reshape(9, *dims[::-1])


def oracle_step(U, axis, recon, second):
    """The middle layer of five: second, mirror image, U, mirror image, second."""
    k = 3 - axis
    F = U.copy()
    F[1 + axis] *= -1
    F[5 + axis] *= -1
    V = np.concatenate([second(F), F, U, F, second(F)], axis=k)
    o = O.OracleState(V.shape[:0:-1], 0.1, dtype=np.float64, recon=recon)
    o.set_conserved(V.reshape(9, -1))
    o.step(DT, ch=CH)
    return np.take(np.asarray(o.U).reshape(V.shape), [2], axis=k)


@pytest.mark.parametrize("recon", ["plm", "ppm"])
@pytest.mark.parametrize("dims", [(8, 1, 6), (1, 4, 5), (6, 7, 1)])
def test_the_second_ghost_layer_matters(dims, recon):
    """The check's own check: a second layer read from the next cell of the field changes the step."""
    U, axis = conserved(dims), dims.index(1)
    right = oracle_step(U, axis, recon, lambda F: F)
    wrong = oracle_step(U, axis, recon, lambda F: np.roll(F, 1, axis=3 if axis != 0 else 2))
    assert np.abs(right - wrong).max() > 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 1e-5)])
@pytest.mark.parametrize("recon", ["plm", "ppm"])
@pytest.mark.parametrize("dims", [(8, 1, 6), (1, 4, 5), (6, 7, 1)])
def test_step_mirrors_the_cell_into_both_layers(dims, recon, dtype, tol):
    """The repository's bars for one step (1e-12 and 1e-5), of each field's maximum."""
    U, axis = conserved(dims).astype(dtype), dims.index(1)
    bcs = tuple("reflecting" if d == axis else "periodic" for d in range(3))
    s = M.allocate_state(dims, 0.1, dtype=dtype, recon=recon, bcs=bcs)
    s.set_conserved(U.reshape(9, -1))
    M.step(s, DT, ch=CH)
    want = oracle_step(U.astype(np.float64), axis, recon, lambda F: F).reshape(9, -1)
    got = s.conserved().astype(np.float64)
    for v in range(9):
        assert np.abs(got[v] - want[v]).max() <= tol * np.abs(want[v]).max(), v
