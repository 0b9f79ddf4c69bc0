"""The HLLD solver's star-flux form and its guarded form on faces at the line between them,
against the float64 oracle (glm_physics.jl:255-307)."""
import numpy as np
import pytest

import oracle as O
import pmfmhd as M

pytestmark = pytest.mark.gpu


def faces(kind, n=256):
    rng = np.random.default_rng(11)

    def side():
        q = np.zeros((n, 9))
        q[:, 0] = np.exp(rng.normal(0, 0.5, n))
        q[:, 1:4] = rng.normal(0, 0.5, (n, 3))
        q[:, 4] = np.exp(rng.normal(0, 0.5, n))
        q[:, 5:8] = rng.normal(0, 0.7, (n, 3))
        q[:, 8] = rng.normal(0, 0.1, n)
        return q

    L, R = side(), side()
    if kind == "supersonic":  # an outer wave clamped at zero, either way
        for q in (L, R):
            q[:, 1:4] += np.where(np.arange(n) % 2, 6.0, -6.0)[:, None]
    elif kind == "zero_field":
        L[:, 5:8] = R[:, 5:8] = 0.0
        L[:, 8] = R[:, 8] = 0.0
    elif kind == "guarded_lanes":  # |denK| below 1e-12 on every third face of a wave
        k = np.arange(n) % 3 == 0
        for q in (L, R):
            q[k, 1:4] = 1e-8 * rng.normal(0, 1, (k.sum(), 3))
            q[k, 4] = 1e-14
            q[k, 5:9] = 1e-8 * rng.normal(0, 1, (k.sum(), 4))
            q[k, 0] = 1.0
    return L, R


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["ordinary", "supersonic", "zero_field", "guarded_lanes"])
def test_hlld_forms_match_oracle(kind, dtype):
    """float64: 1e-12 of each component's scale, as the other parity tests; float32: 64 roundings
    of it (a face is some 60 dependent operations), or four times the float32 oracle's own error."""
    L, R = faces(kind)
    kw = dict(llf_dmin=0.0, smallr=1e-12, pfl=1e-20)
    L, R = L.astype(dtype), R.astype(dtype)
    for d in range(3):
        want = O.riemann_batch(L.astype(np.float64), R.astype(np.float64), d, 1.5, riemann="hlld", **kw)
        s = M.allocate_state((4, 4, 4), 0.25, dtype=dtype, riemann="hlld", **kw)
        got = M.riemann_flux(s, L, R, d, ch=1.5).astype(np.float64)
        assert np.all(np.isfinite(got))
        scale = np.maximum(np.abs(want).max(axis=0), 1e-30)
        err = (np.abs(got - want) / scale).max(axis=1)
        if dtype == np.float64:
            assert err.max() < 1e-12, (kind, d)
        else:
            own = O.riemann_batch(L, R, d, 1.5, dtype=np.float32, riemann="hlld", **kw).astype(np.float64)
            bound = np.maximum(64 * 2.0 ** -24, 4 * (np.abs(own - want) / scale).max(axis=1))
            assert np.all(err <= bound), (kind, d, err.max())
