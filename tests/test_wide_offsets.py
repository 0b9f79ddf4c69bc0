"""The 64-bit-offset instances of the step kernels (fields of 4 GiB and more), forced onto small
grids, against the 32-bit-offset ones: source terms, boundaries, float64, the surrogate."""
import os

import numpy as np
import pytest

import pmfmhd as M
from pmfmhd.surrogate import Surrogate, step_surrogate
from test_ref_dispatch import state

pytestmark = pytest.mark.gpu
WEIGHTS = os.path.join(os.path.dirname(M.__file__), "data", "surrogate_weights.npy")


def narrow_and_wide(monkeypatch, dims, dtype, run, **kw):
    out = []
    for wide in ("0", "1"):
        monkeypatch.setenv("PMFMHD_WIDE_OFFSETS", wide)
        s = state(dims, dtype, **kw)
        run(s)
        out.append((s.conserved(), M.max_wavespeed(s)))
    assert np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("bcs", [("periodic",) * 3, ("outflow", "reflecting", "periodic")])
@pytest.mark.parametrize("dims", [(16, 12, 4), (33, 13, 9), (5, 3, 2)])
@pytest.mark.parametrize("recon", ["plm_minmod", "plm", "ppm"])
def test_wide_offsets_equal_narrow_offsets(dims, bcs, dtype, recon, monkeypatch):
    corr = np.zeros((9, int(np.prod(dims))))
    corr[1:4] = 0.01 * np.random.default_rng(8).normal(size=(3, corr.shape[1]))

    def run(s):
        M.step(s, 2e-3, ch=3.0, integrator="cube")
        M.step_drag(s, 2e-3, 3.0, 0.98, 0.2, integrator="cube")
        buf = M.correction_buffer(s, corr)
        M.load_psi(s, buf)
        M.step_radiation(s, 2e-3, 3.0, 0.98, 0.2, buf)

    narrow_and_wide(monkeypatch, dims, dtype, run, recon=recon, bcs=bcs)


@pytest.mark.parametrize("dims", [(16, 12, 4), (48, 13, 9)])
def test_surrogate_wide_offsets_equal_narrow_offsets(dims, monkeypatch):
    def run(s):
        net = Surrogate(s, seed=1)
        net.set_weights(np.load(WEIGHTS))
        step_surrogate(s, net, 2e-3, 3.0, thr=0.2)

    narrow_and_wide(monkeypatch, dims, np.float32, run, recon="plm_minmod")
