"""The faces that the HLLD solver sends to its guarded form (a star density below 1e-12, a
degenerate star state: glm_physics.jl:255-307) or to LLF, among ordinary faces of the same wave,
each against the float64 oracle on the scale of its own flux."""
import numpy as np
import pytest

import oracle as O
import pmfmhd as M

CH, G = 1.5, 5.0 / 3.0


def faces(kind, n=256):
    rng = np.random.default_rng(17)
    q = np.zeros((2, n, 9))
    q[..., 0] = np.exp(rng.normal(0, 0.5, (2, n)))
    q[..., 1:4] = rng.normal(0, 0.5, (2, n, 3))
    q[..., 4] = np.exp(rng.normal(0, 0.5, (2, n)))
    q[..., 5:8] = rng.normal(0, 0.7, (2, n, 3))
    q[..., 8] = rng.normal(0, 0.1, (2, n))
    k = np.arange(n) % 3 == 0
    m = k.sum()
    if kind == "degenerate":  # waves of 1e-8 around a unit density: denK of 1e-16
        q[:, k, 0] = 1.0
        q[:, k, 1:4] = 1e-8 * rng.normal(0, 1, (2, m, 3))
        q[:, k, 4] = 1e-14
        q[:, k, 5:9] = 1e-8 * rng.normal(0, 1, (2, m, 4))
    else:  # "thin": densities of 2e-13, moderate waves (pressure and field scaled with the density)
        q[:, k, 0] *= 2e-13
        q[:, k, 4] *= 2e-13
        q[:, k, 5:9] *= 2e-13 ** 0.5
    low = ~k & (np.arange(n) % 5 == 1) & (kind == "degenerate")  # below llf_dmin on one side
    q[0, low, 0] = 5e-5
    return q[0], q[1], k, low


def star(L, R, d):
    """Normal-frame star densities and star-state denominators of either side, and the scale of
    each flux component, in float64."""
    f = [[q[:, 1 + d], q[:, 5 + d]] for q in (L, R)]
    bn = 0.5 * (f[0][1] + f[1][1]) - 0.5 * (R[:, 8] - L[:, 8]) / CH
    b2 = [bn ** 2 + (q[:, 5:8] ** 2).sum(1) - q[:, 5 + d] ** 2 for q in (L, R)]
    pt = [q[:, 4] + 0.5 * b for q, b in zip((L, R), b2)]
    cf = []
    for q, b in zip((L, R), b2):
        c2, s = G * q[:, 4] / q[:, 0], b / q[:, 0] + G * q[:, 4] / q[:, 0]
        cf.append(np.sqrt(0.5 * (s + np.sqrt(np.maximum(s * s - 4 * c2 * bn ** 2 / q[:, 0], 0)))))
    c = np.maximum(*cf)
    u = [a[0] for a in f]
    S = [np.minimum(np.minimum(*u) - c, 0), np.maximum(np.maximum(*u) + c, 0)]
    a = [(S[k] - u[k]) * q[:, 0] for k, q in enumerate((L, R))]
    SM = (a[1] * u[1] - a[0] * u[0] - pt[1] + pt[0]) / (a[1] - a[0])
    rho = [a[k] / (S[k] - SM) for k in range(2)]
    den = [a[k] * (S[k] - SM) - bn ** 2 for k in range(2)]
    v = np.maximum(np.abs(L[:, 1:4]).max(1), np.abs(R[:, 1:4]).max(1)) + c
    d_, p_, B = np.maximum(L[:, 0], R[:, 0]), np.maximum(*pt), np.sqrt(np.maximum(*b2))
    scale = np.empty_like(L)
    scale[:, 0], scale[:, 1:4], scale[:, 4] = d_ * v, (d_ * v * v + p_)[:, None], (d_ * v * v + p_) * v
    scale[:, 5:8], scale[:, 8] = (B * v)[:, None], CH * CH * B
    psi = np.maximum(np.abs(L[:, 8]), np.abs(R[:, 8])) + CH * np.abs(f[0][1] - f[1][1])
    scale[:, 5 + d], scale[:, 8] = psi, CH * CH * (np.abs(f[0][1]) + np.abs(f[1][1])) + CH * psi
    return rho, den, scale


@pytest.mark.parametrize("kind", ["degenerate", "thin"])
def test_the_chosen_faces_are_guarded(kind):
    L, R, k, low = faces(kind)
    assert k.sum() > 80 and (low.sum() > 20) == (kind == "degenerate")
    for d in range(3):
        rho, den, _ = star(L, R, d)
        hit = np.abs(np.array(den)) < 1e-12 if kind == "degenerate" else np.array(rho) < 1e-12
        assert hit[:, k].any(0).all()
        assert not ((np.abs(np.array(den)) < 1e-12) | (np.array(rho) < 1e-12))[:, ~k & ~low].any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["degenerate", "thin"])
def test_guarded_faces_match_oracle_on_their_own_scale(kind, dtype):
    """float64: 1e-12 of the face's own scale, as the other parity tests of theirs; float32: 64
    roundings of it (a face is some 60 dependent operations), or four times the float32 oracle's
    own error."""
    L, R, _, _ = faces(kind)
    kw = dict(llf_dmin=1e-4 if kind == "degenerate" else 0.0, smallr=1e-14, pfl=1e-30)
    L, R = L.astype(dtype), R.astype(dtype)
    L64, R64 = L.astype(np.float64), R.astype(np.float64)
    for d in range(3):
        want = O.riemann_batch(L64, R64, d, CH, riemann="hlld", **kw)
        s = M.allocate_state((4, 4, 4), 0.25, dtype=dtype, riemann="hlld", **kw)
        got = M.riemann_flux(s, L, R, d, ch=CH).astype(np.float64)
        err = np.abs(got - want) / star(L64, R64, d)[2]
        assert np.all(np.isfinite(got))
        if dtype == np.float64:
            assert err.max() < 1e-12, (d, err.max(0))
        else:
            own = np.abs(O.riemann_batch(L, R, d, CH, dtype=np.float32, riemann="hlld", **kw) - want)
            own = own / star(L64, R64, d)[2]
            bound = np.maximum(64 * 2.0 ** -24, 4 * own.max(1, keepdims=True))
            assert np.all(err <= bound), (d, (err / bound).max(0))
