"""GLM steps of the :ref integrator on the fused kernel against the per-cell kernel."""
import numpy as np
import pytest

import pmfmhd as M
from pmfmhd import problems as P

pytestmark = pytest.mark.gpu


def state(dims, dtype, **kw):
    rng = np.random.default_rng(4)
    n = int(np.prod(dims))
    one = np.ones(n)
    q = [one + 0.2 * rng.uniform(-1, 1, n), *rng.normal(0, 0.3, (3, n)), one, *rng.normal(0, 0.4, (3, n)),
         rng.normal(0, 0.05, n)]
    s = M.allocate_state(dims, 0.1, dtype=dtype, **kw)
    s.set_conserved(P.prim2cons(q, 5.0 / 3.0))
    return s


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 2e-6)])
@pytest.mark.parametrize("bcs", [("periodic",) * 3, ("outflow", "reflecting", "periodic")])
@pytest.mark.parametrize("dims", [(16, 12, 4), (19, 14, 9), (5, 3, 2)])
@pytest.mark.parametrize("recon,riemann", [("plm", "hlld"), ("ppm", "hlld"), ("plm_minmod", "hll"), ("ppm", "llf")])
def test_ref_step_kernels_agree(dims, bcs, dtype, tol, recon, riemann):
    """Plain, drag (moving target) and radiation steps: the repository's bars for two kernels of one
    scheme (1e-12 / 2e-6 of each field's largest value); PLM plain steps bit for bit; the
    CFL speed kept by the fused step equals a fresh reduction."""
    for kind in ("plain", "drag", "radiation"):
        out = []
        for per_cell in (True, False):
            s = state(dims, dtype, recon=recon, riemann=riemann, bcs=bcs)
            M.set_ct_kernel(s, per_cell)
            corr = np.zeros((9, s.ncells))
            corr[1:4] = 0.01 * np.random.default_rng(8).normal(size=(3, s.ncells))
            buf = M.correction_buffer(s, corr)
            if kind == "plain":
                M.step(s, 2e-3, ch=3.0)
            elif kind == "drag":
                M.step_drag(s, 2e-3, 3.0, 0.98, 0.2, target_velocity=(0.1, -0.2, 0.05))
            else:
                M.load_psi(s, buf)
                M.step_radiation(s, 2e-3, 3.0, 0.98, 0.2, buf)
            kept = M.max_wavespeed(s)
            s.device_ptr(0)  # the next speed is a fresh reduction
            assert M.max_wavespeed(s) == kept
            out.append(s.conserved().astype(np.float64))
        a, b = out
        assert np.all(np.isfinite(b))
        if kind == "plain" and recon != "ppm":
            assert np.array_equal(a, b)
        for v in range(9):
            assert np.abs(a[v] - b[v]).max() <= tol * max(np.abs(a[v]).max(), 1e-3), (kind, v)
