"""The work a user of this library has it do, as cases that can be timed and checked.

A case is one pass through the public entry points: a time step (or a few) of one of the
solvers on the sizes and inputs of the repository's own benchmark, tests and named
configurations, the ensemble, the learned flux and its training. Inputs are made on the
GPU from the seed: random solenoidal fields built from Fourier modes, in the spectra and
amplitudes of ``pmfmhd.problems`` (its host generator takes seconds at 256^3). ``exact``
is the same scheme written out in plain torch at 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pmf-glm_amd"))
import pmfmhd as M  # noqa: E402
from pmfmhd.ensemble import Ensemble  # noqa: E402
from pmfmhd.surrogate import Surrogate, step_surrogate  # noqa: E402

DEV = "cuda"
GAMMA, SMALLR, PFL, LLF_DMIN, GLM_CR = 5.0 / 3.0, 1e-6, 1e-7, 1e-4, 0.18
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(M.__file__)), "data", "surrogate_weights.npy")


def _case(kind, n, name=None, **kw):
    nx, ny, nz = (n, n, n) if isinstance(n, int) else n
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, recon="plm_minmod", riemann="hlld", bc="ppp", dtype="float32",
             integrator="cube", ic="turb", steps=1)
    c.update(kw)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest benchmark configuration (static 32^3), host-driven: read dt back, step.
        # Launches and the round trip per step are what a user of small grids waits for.
        _case("loop", 32, "static_32_host_loop", ic="static", steps=4),
        # the reference's own benchmark: float32 PPM-HLLD on a smooth 128^3 state, step into
        # the caller's arrays
        _case("into", 128, "ppm_128_step_into", recon="ppm", ic="smooth"),
        # the flagship workload: decaying turbulence at 256^3, steps queued with the device's dt
        _case("advance", 256, "turb_256_advance", steps=2),
        # the largest configuration: supersonic 512^3
        _case("into", 512, "mach15_512_step_into", ic="mach15"),
        # step()'s default integrator and default limiter on a ragged grid with boundaries
        _case("into", (200, 125, 83), "default_step_ragged_bounded", recon="plm", bc="orp", integrator="ref"),
        # double precision, for validation runs
        _case("into", 160, "float64_160_step_into", recon="plm", dtype="float64"),
        # constrained transport: the reference's CT benchmark, and the flagship size
        _case("ct", 96, "ct_ppm_96_loop", recon="ppm", integrator="ref", ic="smooth"),
        _case("ct", 256, "ct_256_loop", integrator="ref"),
        # the production step: radiation-coupled update with all residuals tracked, then the
        # two passive species it carries
        _case("coupled", 192, "coupled_192_production_step"),
        # an ensemble of uneven small cubes, each with its own time step
        _case("ensemble", 32, "ensemble_mixed", ic="static", steps=16, n32=16, n64=12, n128=4),
        # the step with the learned flux on smooth faces, at the default gate
        _case("surrogate", 192, "surrogate_192_step", ic="static_large_scale", thr=0.02),
        # training the learned flux: Adam on mini-batches of the trainer's size
        _case("train", 32, "train_batch_8192", steps=8, batch=8192, pairs=1 << 17, lr=1e-4),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["loop", "into", "into", "into", "advance", "ct", "coupled", "ensemble", "surrogate", "train"])
    recon = rng.choice(["plm", "plm_minmod", "ppm"])
    if kind == "loop":
        return _case(kind, (size(16, 96), size(16, 96), size(16, 96)), recon=recon, ic="static", steps=rng.randint(1, 5))
    if kind == "into":
        f64 = rng.random() < 0.25
        n = tuple(size(24, 200 if f64 else 330) for _ in range(3))
        bc = rng.choice(["ppp", "ppp", "ooo", "orp", "rrr", "pro"])
        return _case(kind, n, recon=recon, riemann=rng.choice(["hlld", "hlld", "hll", "llf"]), bc=bc,
                     dtype="float64" if f64 else "float32", integrator=rng.choice(["cube", "ref"]),
                     ic=rng.choice(["turb", "mach15", "smooth"]))
    if kind == "advance":
        return _case(kind, tuple(size(48, 300) for _ in range(3)), recon=recon, steps=rng.randint(1, 4))
    if kind == "ct":
        return _case(kind, tuple(size(32, 256) for _ in range(3)), recon=recon, integrator="ref",
                     riemann=rng.choice(["hlld", "hlld", "hll"]))
    if kind == "coupled":
        return _case(kind, size(32, 220), recon=rng.choice(["plm", "plm_minmod"]))
    if kind == "ensemble":
        return _case(kind, 32, recon=recon, ic="static", steps=rng.randint(4, 16), n32=rng.randint(1, 24),
                     n64=rng.randint(1, 16), n128=rng.randint(0, 4))
    if kind == "surrogate":
        return _case(kind, (16 * rng.randint(2, 13), size(24, 200), size(24, 200)), ic="static_large_scale",
                     thr=round(math.exp(rng.uniform(math.log(0.0025), math.log(0.02))), 5))
    return _case(kind, 32, steps=rng.randint(2, 12), batch=size(1000, 8192), pairs=1 << 17, lr=1e-4)


# ---- inputs -------------------------------------------------------------------------------

def _modes(shape, gen, kmax, index, rms, ncomp, nmodes=256):
    """ncomp real random fields of the (nz, ny, nx) grid: nmodes Fourier modes with 1 <= |m| <= kmax and
    power ~ k^index per mode, together solenoidal under the centred difference when ncomp = 3."""
    nz, ny, nx = shape
    dims = np.array([nx, ny, nz])
    rs = np.random.RandomState(int(torch.randint(0, 1 << 31, (1,), generator=gen)))
    m = rs.randint(-kmax, kmax + 1, (8 * nmodes + 64, 3))
    m = np.where(dims == 1, 0, m)
    k = np.sqrt((m ** 2).sum(1))
    m, k = m[(k >= 1) & (k <= kmax)][:nmodes], k[(k >= 1) & (k <= kmax)][:nmodes]
    c = (rs.randn(len(k), ncomp) + 1j * rs.randn(len(k), ncomp)) * (k ** (0.5 * index))[:, None]
    if ncomp == 3:
        s = np.sin(2 * np.pi * m / dims)
        c = c - s * ((c * s).sum(1) / np.maximum((s * s).sum(1), 1e-30))[:, None]

    def phase(axis, n):
        return torch.from_numpy(np.exp(2j * np.pi * np.outer(np.arange(n), m[:, axis]) / n)).to(DEV, torch.complex64)

    ex, ey, ez = phase(0, nx), phase(1, ny), phase(2, nz)
    zy = (ez[:, None, :] * ey[None, :, :]).reshape(nz * ny, -1)
    out = []
    for d in range(ncomp):
        a = zy * torch.from_numpy(c[:, d]).to(DEV, torch.complex64)
        out.append((a.real.contiguous() @ ex.real.T.contiguous() - a.imag.contiguous() @ ex.imag.T.contiguous())
                   .reshape(shape))
    scale = rms / max(float(torch.stack([(o.double() ** 2).mean() for o in out]).sum().sqrt()), 1e-30)
    return [o * scale for o in out]


def _grid_of(case):
    return case["nz"], case["ny"], case["nx"]


def _generators(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    h = torch.Generator()
    h.manual_seed(seed + 7919)
    return g, h


def _initial(case, shape, seed):
    """Conserved state (9, nz, ny, nx) in the case's precision."""
    dev, gen = _generators(seed)
    n = min(shape)
    ic = case["ic"]
    if ic == "smooth":  # the reference benchmark's smooth state, with the seed's phases
        nz, ny, nx = shape
        p = np.random.RandomState(seed).uniform(0, 2 * np.pi, 6)
        x = (2 * np.pi * (torch.arange(nx, device=DEV) + 0.5) / nx).view(1, 1, nx).expand(shape)
        y = (2 * np.pi * (torch.arange(ny, device=DEV) + 0.5) / ny).view(1, ny, 1).expand(shape)
        z = (2 * np.pi * (torch.arange(nz, device=DEV) + 0.5) / nz).view(nz, 1, 1).expand(shape)
        rho = torch.ones(shape, device=DEV)
        v = [0.2 * torch.sin(z + p[0]), 0.2 * torch.sin(x + p[1]), 0.2 * torch.sin(y + p[2])]
        b = [0.3 + 0.1 * torch.sin(2 * y + p[3]), 0.1 * torch.sin(2 * z + p[4]), 0.1 * torch.sin(2 * x + p[5])]
    else:
        noise = torch.randn(shape, generator=dev, device=DEV)
        static = ic.startswith("static")
        kmax = max(2, n // {"static": 4, "static_large_scale": 32}.get(ic, 8))
        if ic == "mach15":
            rho = torch.exp(0.3 * noise - 0.045)
        else:
            rho = 1 + 0.01 * noise
        b = _modes(shape, gen, kmax, 2.0, 0.3 if static else 1.0, 3)
        if static:
            v = [torch.zeros(shape, device=DEV)] * 3
        else:
            v = _modes(shape, gen, kmax, -2.0, (1.5 if ic == "mach15" else 0.5) * math.sqrt(GAMMA), 3)
    t = torch.float64 if case["dtype"] == "float64" else torch.float32
    rho, v, b = rho.to(t), [a.to(t) for a in v], [a.to(t) for a in b]
    U = torch.empty((9,) + tuple(shape), device=DEV, dtype=t)
    U[0] = rho
    for d in range(3):
        U[1 + d] = rho * v[d]
        U[5 + d] = b[d]
    U[4] = 1.0 / (GAMMA - 1) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + 0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
    U[8] = 0
    return U


def _faces(U, seed):
    """Divergence-free faces near U's cell field (the curl of an edge potential), and U with the face average
    as its cell field and its thermal pressure kept."""
    _, gen = _generators(seed + 1)
    shape = tuple(U.shape[1:])
    rms = float((U[5:8].double() ** 2).sum(0).mean().sqrt())
    A = _modes(shape, gen, max(2, min(shape) // 8), 0.0, 1.0, 3)
    up = lambda a, d: torch.roll(a, -1, 2 - d)  # noqa: E731
    F = torch.stack([(up(A[2], 1) - A[2]) - (up(A[1], 2) - A[1]), (up(A[0], 2) - A[0]) - (up(A[2], 0) - A[2]),
                     (up(A[1], 0) - A[1]) - (up(A[0], 1) - A[0])])
    F = (F * (rms / float((F.double() ** 2).sum(0).mean().sqrt()))).to(U.dtype)
    U = U.clone()
    U[4] -= 0.5 * (U[5:8] ** 2).sum(0)
    for d in range(3):
        U[5 + d] = 0.5 * (F[d] + up(F[d], d))
    U[4] += 0.5 * (U[5:8] ** 2).sum(0)
    return U, F


class _Device:
    """A device allocation of the library, for torch.as_tensor."""

    def __init__(self, owner, ptr, shape, dtype):
        self.owner = owner  # the tensor keeps this object, and with it the allocation
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=np.dtype(dtype).str, data=(int(ptr), False),
                                             version=2)


def _view(owner, ptr, shape, dtype):
    return torch.as_tensor(_Device(owner, ptr, shape, dtype), device=DEV)


def _allocate(case, **kw):
    bcs = tuple({"p": "periodic", "o": "outflow", "r": "reflecting"}[b] for b in case["bc"])
    return M.allocate_state((case["nx"], case["ny"], case["nz"]), 1.0 / case["nx"], dtype=np.dtype(case["dtype"]),
                            recon=case["recon"], riemann=case["riemann"], bcs=bcs, **kw)


def _own_state(case, U, **kw):
    """A library state holding U; its two field sets as tensors (a step writes the other set and swaps)."""
    s = _allocate(case, **kw)
    shape = (9,) + tuple(U.shape[1:])
    sets = [_view(s, s.device_ptr(0), shape, s.dtype), _view(s, s.scratch_ptr(0), shape, s.dtype)]
    sets[0].copy_(U)
    return s, sets


def _pairs(case, seed):
    """Training rows of smooth faces: inputs, HLLD targets, states, as the solver's dump gives them."""
    rs = np.random.RandomState(seed)
    n, thr = case["pairs"], 0.02

    def normal(scale, *shape):
        return torch.from_numpy(rs.standard_normal(shape) * scale)

    mean = [torch.exp(normal(0.1, n)), normal(0.3, n), normal(0.3, n), normal(0.3, n), torch.exp(normal(0.15, n)),
            normal(0.4, n), normal(0.4, n), normal(0.4, n)]
    jump = [normal(0.004, n) * (mean[v] if v in (0, 4) else 1.0) for v in range(8)]
    jump[5] = torch.zeros(n, dtype=torch.float64)
    L = [(m - 0.5 * j).to(DEV) for m, j in zip(mean, jump)] + [torch.zeros(n, device=DEV, dtype=torch.float64)]
    R = [(m + 0.5 * j).to(DEV) for m, j in zip(mean, jump)] + [torch.zeros(n, device=DEV, dtype=torch.float64)]
    x, s, _ = _encode(L, R, thr)
    zero = torch.zeros_like(L[0])
    f = _hlld(L, R, L[5], zero, zero)
    c = _central(L, R)
    y = [(f[k] - c[k]) / s[k] if k not in (5, 8) else zero for k in range(9)]
    S = torch.stack(L[:8] + R[:8] + [zero, zero], 1)
    return tuple(a.float().cpu().numpy() for a in (torch.stack(x, 1), torch.stack(y, 1), S))


def _part_trained(seed):
    """Weights part-way through training: the trained ones with noise."""
    w = np.load(WEIGHTS)
    return (w + 0.05 * np.random.RandomState(seed + 1).standard_normal(w.shape)).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "ensemble":
        edges = [32] * case["n32"] + [64] * case["n64"] + [128] * case["n128"]
        e = Ensemble(edges, recon=case["recon"], riemann=case["riemann"])
        for c, n in enumerate(edges):
            e.upload(c, _initial(case, (n, n, n), seed * 1009 + c).reshape(9, -1).cpu().numpy())
        st.update(e=e, edges=edges)
        return st
    if kind == "train":
        s = M.allocate_state((32, 32, 32), 1 / 32, dtype=np.float32)  # parameters and stream
        net = Surrogate(s, seed=1)
        net.set_weights(_part_trained(seed))
        X, Y, S = _pairs(case, seed)
        net.reserve(len(X))
        net.upload(X, Y, S)
        st.update(s=s, net=net, seed=seed)
        return st
    U = _initial(case, _grid_of(case), seed)
    if kind == "into":
        s = _allocate(case, workspace=True)
        O = torch.empty_like(U)
        smax = _smax(U)
        dx = 1.0 / case["nx"]
        dt = 0.2 * dx / smax
        st.update(s=s, U=U, O=O, pu=[U[v].data_ptr() for v in range(9)], po=[O[v].data_ptr() for v in range(9)],
                  args=(dt, smax, math.exp(-GLM_CR * smax * dt / dx)))
        torch.cuda.synchronize()
        return st
    if kind == "ct":
        U, F = _faces(U, seed)
        s, sets = _own_state(case, U, mhd_solver="ct")
        faces = _view(s, s.ct_ptr(0), F.shape, s.dtype)
        faces.copy_(F)
        st.update(faces=faces)
    else:
        s, sets = _own_state(case, U)
    if kind == "coupled":
        _, gen = _generators(seed + 2)
        n = s.ncells
        corr = M.correction_buffer(s)
        slots = _view(corr, corr.ptr, (9,) + _grid_of(case), s.dtype)
        slots[1:4] = torch.stack(_modes(_grid_of(case), gen, 4, -2.0, 0.01, 3))
        q = [M.DeviceBuffer(4 * n) for _ in range(4)]
        species = [_view(b, b.ptr, _grid_of(case), s.dtype) for b in q[:2]]
        for a, f in zip(species, _fractions(_grid_of(case), seed)):
            a.copy_(U[0] * f)
        st.update(corr=corr, slots=slots, q=q, species=species)
    if kind == "surrogate":
        net = Surrogate(s, seed=0)
        net.set_weights(np.load(WEIGHTS))
        st.update(net=net)
    st.update(s=s, sets=sets, done=0)
    torch.cuda.synchronize()
    return st


def _fractions(shape, seed):
    """Two mass fractions (an ion fraction and a smaller molecular one)."""
    _, gen = _generators(seed + 3)
    a, b = _modes(shape, gen, 8, -2.0, 1.0, 2)
    return 0.4 + 0.1 * torch.tanh(a), 0.05 + 0.02 * torch.tanh(b)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "into":
        dt, ch, decay = st["args"]
        M.step_into(st["s"], st["pu"], st["po"], dt, ch, decay, integrator=case["integrator"])
        return st["O"]
    if kind == "ensemble":
        e = st["e"]
        e.run(case["steps"])
        # the ensemble hands its members out as host arrays: two of them are read each pass
        return [e.download(c) for c in _some(st["edges"])]
    if kind == "train":
        losses = st["net"].train(case["steps"], batch=case["batch"], lr=case["lr"], seed=st["seed"])
        # float32: what the losses are computed in
        return dict(weights=st["net"].weights(), losses=losses.astype(np.float32))
    s = st["s"]
    out = {}
    if kind == "advance":
        M.advance(s, case["steps"], cfl=0.2)
    for _ in range(case["steps"] if kind != "advance" else 0):
        dt, smax = M.compute_dt(s, 0.2)
        if kind == "loop":
            M.step(s, float(dt), ch=float(smax), integrator=case["integrator"])
        elif kind == "ct":
            M.step(s, float(dt), integrator="ref")
            out["faces"] = st["faces"]
        elif kind == "surrogate":
            step_surrogate(s, st["net"], float(dt), float(smax), thr=case["thr"])
        else:
            q = st["q"]
            M.species_to_fractions(s, q[0], q[1])
            M.load_psi(s, st["corr"])
            M.step_radiation(s, float(dt), float(smax), 0.99, 0.1, st["corr"], integrator="cube")
            M.advect_species(s, q[0], q[2], float(dt), species2=q[1], scratch2=q[3])
            # the remainders in slots 5-8 are rounding errors: they have no value of their own
            out.update(density_perturbation=st["slots"][4], species1=st["species"][0], species2=st["species"][1])
    st["done"] += case["steps"]
    out["fields"] = st["sets"][st["done"] & 1]
    return out


def _some(edges):
    """The members that a pass reads out: one of each of the two smaller edges."""
    return sorted({n: c for c, n in enumerate(edges) if n <= 64}.values())


# ---- what a pass cannot do without --------------------------------------------------------

def work(case):
    kind = case["kind"]
    cells = case["nx"] * case["ny"] * case["nz"]
    size = 8 if case["dtype"] == "float64" else 4
    # operations of one cell-update: one prediction, three faces, the update and its CFL speed
    flops = {"hlld": 1400, "hll": 1000, "llf": 1000}[case["riemann"]] * cells * case["steps"]
    bytes_ = 18 * size * cells * case["steps"]
    if kind == "ct":
        bytes_ = 24 * size * cells * case["steps"]
    elif kind == "coupled":  # psi and three corrections in, five residuals in and out, two species in and out
        bytes_ = (18 + 4 + 10 + 4) * size * cells
    elif kind == "ensemble":
        cells = case["n32"] * 32 ** 3 + case["n64"] * 64 ** 3 + case["n128"] * 128 ** 3
        bytes_, flops = 18 * size * cells * case["steps"], 1400 * cells * case["steps"]
    elif kind == "surrogate":  # most faces go through the network: 9993 parameters each
        flops += 3 * cells * 2 * 9993
    elif kind == "train":  # forward, input gradients and weight gradients
        flops = case["steps"] * case["batch"] * 3 * 2 * 9993
        bytes_ = case["steps"] * (case["batch"] * 100 + 9993 * 28)
    return {"bytes": bytes_, "flops": flops}


# ---- the scheme at 64 bits ----------------------------------------------------------------

def _smax(U):
    q = _prim(U.double())
    return float(max((q[1 + d].abs() + _cfast(q, 5 + d)).max() for d in range(3)))


def _prim(U):
    rho = U[0].clamp(min=SMALLR)
    p = (GAMMA - 1) * (U[4] - 0.5 * (U[1] ** 2 + U[2] ** 2 + U[3] ** 2) / rho - 0.5 * (U[5] ** 2 + U[6] ** 2 + U[7] ** 2))
    return [rho, U[1] / rho, U[2] / rho, U[3] / rho, p.clamp(min=PFL), U[5], U[6], U[7], U[8]]


def _cons(q):
    return [q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3],
            q[4] / (GAMMA - 1) + 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)
            + 0.5 * (q[5] ** 2 + q[6] ** 2 + q[7] ** 2), q[5], q[6], q[7], q[8]]


def _cfast(q, n):
    c2 = GAMMA * q[4] / q[0]
    d2 = 0.5 * ((q[5] ** 2 + q[6] ** 2 + q[7] ** 2) / q[0] + c2)
    return (d2 + (d2 * d2 - c2 * q[n] ** 2 / q[0]).clamp(min=0).sqrt()).sqrt()


def _flux(q):
    """Physical flux along the first axis of a normal-frame state; the GLM slots are zero."""
    rho, u, v, w, p, bn, by, bz = q[:8]
    pt = p + 0.5 * (bn * bn + by * by + bz * bz)
    E = _cons(q)[4]
    z = torch.zeros_like(rho)
    return [rho * u, rho * u * u + pt - bn * bn, rho * u * v - bn * by, rho * u * w - bn * bz,
            (E + pt) * u - bn * (u * bn + v * by + w * bz), z, u * by - v * bn, u * bz - w * bn, z]


def _frame(q, d):
    n, a, b = d, (d + 1) % 3, (d + 2) % 3
    return [q[0], q[1 + n], q[1 + a], q[1 + b], q[4], q[5 + n], q[5 + a], q[5 + b], q[8]]


def _unframe(f, d):
    n, a, b = d, (d + 1) % 3, (d + 2) % 3
    F = [None] * 9
    F[0], F[4], F[8] = f[0], f[4], f[8]
    F[1 + n], F[1 + a], F[1 + b] = f[1], f[2], f[3]
    F[5 + n], F[5 + a], F[5 + b] = f[5], f[6], f[7]
    return F


def _hlld(L, R, bn, fbn, fpsi):
    cmax = torch.maximum(_cfast(L, 5), _cfast(R, 5))
    S = [(torch.minimum(L[1], R[1]) - cmax).clamp(max=0), (torch.maximum(L[1], R[1]) + cmax).clamp(min=0)]
    pt = [q[4] + 0.5 * (bn * bn + q[6] ** 2 + q[7] ** 2) for q in (L, R)]
    a = [(S[0] - L[1]) * L[0], (S[1] - R[1]) * R[0]]
    SM = (a[1] * R[1] - a[0] * L[1] - pt[1] + pt[0]) / (a[1] - a[0])
    pts = (a[1] * pt[0] - a[0] * pt[1] + a[0] * a[1] * (R[1] - L[1])) / (a[1] - a[0])
    star = []
    for k, q in enumerate((L, R)):
        ds = (a[k] / (S[k] - SM)).clamp(min=1e-12)
        den = a[k] * (S[k] - SM) - bn * bn
        deg = den.abs() < 1e-12
        den = torch.where(deg, torch.ones_like(den), den)
        fac = torch.where(deg, torch.zeros_like(den), bn * (SM - q[1]) / den)
        gg = torch.where(deg, torch.ones_like(den), (a[k] * (S[k] - q[1]) - bn * bn) / den)
        v, w, by, bz = q[2] - q[6] * fac, q[3] - q[7] * fac, q[6] * gg, q[7] * gg
        vb, vbs = q[1] * bn + q[2] * q[6] + q[3] * q[7], SM * bn + v * by + w * bz
        E = _cons(list(q[:5]) + [bn, q[6], q[7], q[8]])[4]
        Es = ((S[k] - q[1]) * E - pt[k] * q[1] + pts * SM + bn * (vb - vbs)) / (S[k] - SM)
        star.append((ds, v, w, by, bz, E, Es, vbs))
    sq = [s[0].sqrt() for s in star]
    Ss = [SM - bn.abs() / sq[0], SM + bn.abs() / sq[1]]
    sg = torch.where(bn >= 0, 1.0, -1.0).to(bn.dtype)
    den = sq[0] + sq[1]
    vyss = (sq[0] * star[0][1] + sq[1] * star[1][1] + (star[1][3] - star[0][3]) * sg) / den
    vzss = (sq[0] * star[0][2] + sq[1] * star[1][2] + (star[1][4] - star[0][4]) * sg) / den
    byss = (sq[0] * star[1][3] + sq[1] * star[0][3] + sq[0] * sq[1] * (star[1][1] - star[0][1]) * sg) / den
    bzss = (sq[0] * star[1][4] + sq[1] * star[0][4] + sq[0] * sq[1] * (star[1][2] - star[0][2]) * sg) / den
    vbss = SM * bn + vyss * byss + vzss * bzss
    out = []
    for k, q in enumerate((L, R)):
        ds, v, w, by, bz, E, Es, vbs = star[k]
        Ess = Es + (-1 if k == 0 else 1) * sq[k] * (vbs - vbss) * sg
        inner = (Ss[0] < 0) if k == 0 else (Ss[1] >= 0)
        c = torch.where(inner, Ss[k], torch.zeros_like(SM))
        F = _flux(list(q[:5]) + [bn, q[6], q[7], q[8]])
        out.append([F[0] + S[k] * (ds - q[0]), F[1] + S[k] * (ds * SM - q[0] * q[1]),
                    F[2] + S[k] * (ds * v - q[0] * q[2]) + c * ds * (vyss - v),
                    F[3] + S[k] * (ds * w - q[0] * q[3]) + c * ds * (vzss - w),
                    F[4] + S[k] * (Es - E) + c * (Ess - Es), None,
                    F[6] + S[k] * (by - q[6]) + c * (byss - by), F[7] + S[k] * (bz - q[7]) + c * (bzss - bz)])
    left = SM >= 0
    f = [None if out[0][i] is None else torch.where(left, out[0][i], out[1][i]) for i in range(8)]
    f[5] = fbn
    return f + [fpsi]


def _two_wave(L, R, riemann, ch, bn, fbn, fpsi):
    L, R = list(L[:5]) + [bn] + list(L[6:]), list(R[:5]) + [bn] + list(R[6:])
    cL, cR, fL, fR, uL, uR = _cfast(L, 5), _cfast(R, 5), _flux(L), _flux(R), _cons(L), _cons(R)
    if riemann == "hll":
        SL = torch.minimum(L[1] - cL, R[1] - cR).clamp(max=0)
        SR = torch.maximum(L[1] + cL, R[1] + cR).clamp(min=0)
        f = [(SR * fL[i] - SL * fR[i] + SL * SR * (uR[i] - uL[i])) / (SR - SL) for i in range(9)]
    else:
        s = torch.maximum(L[1].abs() + cL, R[1].abs() + cR).clamp(min=ch)
        f = [0.5 * (fL[i] + fR[i]) - 0.5 * s * (uR[i] - uL[i]) for i in range(9)]
    f[5], f[8] = fbn, fpsi
    return f


def _encode(L, R, thr):
    """The learned flux's 16 inputs, its output scales and its gate."""
    m = [0.5 * (a + b) for a, b in zip(L, R)]
    a2 = (GAMMA * m[4] + L[5] ** 2 + m[6] ** 2 + m[7] ** 2) / m[0]
    a, sr = a2.sqrt(), m[0].sqrt()
    sc = [m[0], a, a, a, m[0] * a2, a * sr, a * sr, a * sr]
    m[5] = 0.5 * (L[5] + R[5])
    x = []
    for v in range(8):
        x += [m[v] / sc[v], (R[v] - L[v]) / (2 * thr * sc[v])]
    z = torch.zeros_like(a)
    s = [thr * m[0] * a] + [thr * m[0] * a2] * 3 + [thr * m[0] * a2 * a, z, thr * a2 * sr, thr * a2 * sr, z]
    bL, bR = [(L[5] ** 2 + q[6] ** 2 + q[7] ** 2).sqrt() for q in (L, R)]
    gate = ((R[0] - L[0]).abs() < thr * m[0]) & ((R[4] - L[4]).abs() < thr * m[4]) & ((bR - bL).abs() <= 0.5 * thr * (bL + bR))
    return x, s, gate


def _central(L, R):
    return [0.5 * (a + b) for a, b in zip(_flux(L), _flux(R))]


def _layers(w):
    out, at = [], 0
    for i, o in ((16, 64), (64, 64), (64, 64), (64, 9)):
        out.append((w[at:at + i * o].reshape(i, o), w[at + i * o:at + i * o + o]))
        at += i * o + o
    return out


def _bf16(a):
    """The network's operands are bfloat16 by definition."""
    return a.float().bfloat16().double()


def _net(w, x, kept=None):
    for k, (W, b) in enumerate(_layers(w)):
        z = _bf16(x) @ _bf16(W) + b
        if kept is not None:
            kept.append((x, z))
        x = torch.nn.functional.gelu(z, approximate="tanh") if k < 3 else z
    return x


def _gradient(w, x, target):
    """Mean squared error over the learned outputs and its gradient."""
    kept = []
    d = _net(w, x, kept) - target
    d[:, [5, 8]] = 0
    n = 7.0 * len(x)
    dz, g = 2 * d / n, []
    for (W, _), (a, _), below in zip(reversed(_layers(w)), reversed(kept), [*reversed(kept[:-1]), None]):
        g = [(_bf16(a).T @ _bf16(dz)).reshape(-1), dz.sum(0)] + g
        if below is not None:
            z = below[1]
            u = 0.7978845608028654 * (z + 0.044715 * z ** 3)
            s = torch.sigmoid(2 * u)
            slope = s + 2 * z * s * (1 - s) * 0.7978845608028654 * (1 + 3 * 0.044715 * z * z)
            dz = (_bf16(dz) @ _bf16(W).T) * slope
    return float((d * d).sum() / n), torch.cat(g)


def _riemann(L, R, case, ch, face=None, net=None):
    """Normal-frame flux of the case's solver: GLM, or with the CT face field, or with the learned flux."""
    L, R = list(L), list(R)
    for q in (L, R):
        q[0], q[4] = q[0].clamp(min=SMALLR), q[4].clamp(min=PFL)
    if face is not None:
        bn, fbn, fpsi, ch = face, torch.zeros_like(face), torch.zeros_like(face), 0.0
    else:
        bn = 0.5 * (L[5] + R[5]) - 0.5 * (R[8] - L[8]) / ch
        fbn = 0.5 * (L[8] + R[8]) - 0.5 * ch * (R[5] - L[5])
        fpsi = ch * ch * bn
    L[5] = R[5] = bn
    if case["riemann"] != "hlld":
        return _two_wave(L, R, case["riemann"], ch, bn, fbn, fpsi)
    f = _hlld(L, R, bn, fbn, fpsi)
    low = torch.minimum(L[0], R[0]) < LLF_DMIN
    if bool(low.any()):
        f = [torch.where(low, a, b) for a, b in zip(_two_wave(L, R, "llf", ch, bn, fbn, fpsi), f)]
    if net is not None:
        w, thr = net
        x, s, gate = _encode(L, R, thr)
        gate = gate & ~low
        c = _central(L, R)
        y = _net(w, torch.stack([a[gate] for a in x], 1))
        for k in (0, 1, 2, 3, 4, 6, 7):
            f[k][gate] = c[k][gate] + s[k][gate] * y[:, k]
    return f


def _offsets(qm, q0, qp, recon):
    dl, dr = q0 - qm, qp - q0
    z = torch.zeros_like(q0)
    mm = torch.where(dl * dr > 0, torch.sign(dl) * torch.minimum(dl.abs(), dr.abs()), z)
    if recon == "plm_minmod":
        return -0.5 * mm, 0.5 * mm
    if recon == "plm":
        c = 0.5 * (dl + dr)
        s = torch.where(dl * dr > 0, torch.sign(c) * torch.minimum(2 * mm.abs(), c.abs()), z)
        return -0.5 * s, 0.5 * s
    a = 0.25 * (qp - qm) + (qm - 2 * q0 + qp) / 12
    b = 0.25 * (qp - qm) - (qm - 2 * q0 + qp) / 12
    flat = a * b <= 0
    hi = torch.where(a.abs() > 2 * b.abs(), 2 * b, a)
    lo = torch.where(b.abs() > 2 * a.abs(), 2 * a, b)
    return torch.where(flat, z, -lo), torch.where(flat, z, hi)


def _pad(U, bc, z0, z1):
    """Planes z0-2 .. z1+2 of U with two ghost layers in every direction."""
    for d in (2, 1, 0):
        n = U.shape[3 - d]
        i = torch.arange(z0 - 2, z1 + 2) if d == 2 else torch.arange(-2, n + 2)
        if bc[d] == "p":
            j, flip = i % n, None
        elif bc[d] == "o":
            j, flip = i.clamp(0, n - 1), None
        else:
            out = (i < 0) | (i >= n)
            j = torch.where(i < 0, -1 - i, torch.where(i >= n, 2 * n - 1 - i, i))
            flip = torch.where(out, -1.0, 1.0).to(U)
        U = U.index_select(3 - d, j.to(U.device))
        if flip is not None:
            flip = flip.view([-1 if k == 2 - d else 1 for k in range(3)])
            U[1 + d] *= flip
            U[5 + d] *= flip
    return U


def _slab(case, U, z0, z1, dtdx, ch, faces=None, net=None, drag=None, corr=None):
    """The flux divergence of planes z0 .. z1 of a 64-bit state; with CT faces also the face fluxes and EMFs."""
    P = _prim(_pad(U, case["bc"], z0, z1))

    def cut(a, d, lo, ring):  # one cell in from the padded edge (ring: two), moved by lo along axis d
        w = [slice(ring, a.shape[k] - ring) for k in range(3)]
        k = 2 - d
        w[k] = slice(ring + lo, a.shape[k] - ring + lo)
        return a[tuple(w)]

    m0 = [cut(a, 0, 0, 1) for a in P]
    off = [[_offsets(cut(a, d, -1, 1), cut(a, d, 0, 1), cut(a, d, 1, 1), case["recon"]) for a in P] for d in range(3)]
    uh = _cons(m0)
    for d in range(3):
        fp = _unframe(_flux(_frame([a + o[1] for a, o in zip(m0, off[d])], d)), d)
        fm = _unframe(_flux(_frame([a + o[0] for a, o in zip(m0, off[d])], d)), d)
        uh = [u - 0.5 * dtdx * (p - m) for u, p, m in zip(uh, fp, fm)]
    mh = _prim(uh)

    def state(d, side):
        q = [a + o[side] for a, o in zip(mh, off[d])]
        if drag is not None:
            decay, phi1 = drag
            for c in range(3):
                f0 = m0[1 + c] + off[d][1 + c][side]
                q[1 + c] = decay * f0 + phi1 * (q[1 + c] - f0) + corr[c]
        return q

    div = [0.0] * 9
    flux = []
    for d in range(3):
        k = 2 - d
        n = m0[0].shape[k]

        def face(a, first):  # states of the cells below (first = 0) and above (1) the n - 1 faces along d
            w = [slice(1, a.shape[j] - 1) for j in range(3)]
            w[k] = slice(first, n - 1 + first)
            return a[tuple(w)]

        L = [face(a, 0) for a in state(d, 1)]
        R = [face(a, 1) for a in state(d, 0)]
        bn = None if faces is None else torch.cat([faces[d], faces[d].narrow(k, 0, 1)], k)
        F = _unframe(_riemann(_frame(L, d), _frame(R, d), case, ch, bn, net), d)
        div = [s + (f.narrow(k, 0, n - 2) - f.narrow(k, 1, n - 2)) for s, f in zip(div, F)]
        if faces is not None:
            flux.append([f.narrow(k, 0, n - 2) for f in F])
        del L, R, F
    if faces is None:
        return div
    c = [cut(a, 0, 0, 1) for a in mh]
    b = [cut(a, 0, 0, 1) for a in m0]
    emf = [c[3] * b[6] - c[2] * b[7], c[1] * b[7] - c[3] * b[5], c[2] * b[5] - c[1] * b[6]]
    return div, flux, emf


def _step(case, U, dt, ch, decay, dx, net=None):
    """One GLM step of a 64-bit (9, nz, ny, nx) state."""
    out = torch.empty_like(U)
    nz = U.shape[1]
    planes = max(1, (1 << 22) // (U.shape[2] * U.shape[3]))
    for z0 in range(0, nz, planes):
        z1 = min(nz, z0 + planes)
        for v, d in enumerate(_slab(case, U, z0, z1, dt / dx, ch, net=net)):
            out[v, z0:z1] = U[v, z0:z1] + dt / dx * d
    out[8] *= decay
    return out


def _rule(U, dx):
    smax = _smax(U)
    dt = 0.2 * dx / smax
    return dt, smax, math.exp(-GLM_CR * smax * dt / dx)


def _upwind(m, lo, hi):
    return torch.where(m > 0, lo, torch.where(m < 0, hi, 0.5 * (lo + hi)))


def _ct_step(case, U, B, dt, dx):
    """One constrained-transport step: the cell update, upwind edge EMFs, the faces' curl, the cell average."""
    div, flux, emf = _slab(case, U, 0, U.shape[1], dt / dx, 0.0, faces=B)
    U = torch.stack([u + dt / dx * d for u, d in zip(U, div)])
    dn = lambda a, d: torch.roll(a, 1, 2 - d)  # noqa: E731
    up = lambda a, d: torch.roll(a, -1, 2 - d)  # noqa: E731
    edge = [None] * 3
    for e in range(3):
        a, b = (e + 1) % 3, (e + 2) % 3
        Ea, Eb = -flux[a][5 + b], flux[b][5 + a]  # the edge's EMF on the a- and b-faces beside it
        Eam, Ebm, ma, mb, Er = dn(Ea, b), dn(Eb, a), flux[a][0], flux[b][0], emf[e]
        Erm0, Er0m = dn(Er, a), dn(Er, b)
        Ermm = dn(Erm0, b)
        A1, A3 = _upwind(ma, Erm0 - Ebm, Er - Eb), _upwind(dn(ma, b), Ebm - Ermm, Eb - Er0m)
        B1, B3 = _upwind(mb, Er0m - Eam, Er - Ea), _upwind(dn(mb, a), Eam - Ermm, Ea - Erm0)
        edge[e] = 0.25 * ((Ea + Eam + Eb + Ebm) + (A3 - A1) + (B3 - B1))
    B = torch.stack([B[d] - dt / dx * ((up(edge[(d + 2) % 3], (d + 1) % 3) - edge[(d + 2) % 3])
                                       - (up(edge[(d + 1) % 3], (d + 2) % 3) - edge[(d + 1) % 3])) for d in range(3)])
    for d in range(3):
        U[5 + d] = 0.5 * (B[d] + up(B[d], d))
    U[8] = 0
    return U, B


def _ring(a):
    """A field with one periodic ghost layer."""
    for k in range(3):
        n = a.shape[k]
        a = torch.cat([a.narrow(k, n - 1, 1), a, a.narrow(k, 0, 1)], k)
    return a


def _coupled_step(case, U, dv, dt, ch, decay, q, dx):
    """One radiation-coupled step: half-step drag on the face states, the velocity correction, the exact drag
    propagator with its energy loss. Returns the state and the density increment."""
    qh = 0.5 * q
    div = _slab(case, U, 0, U.shape[1], dt / dx, ch, drag=(math.exp(-qh), -math.expm1(-qh) / qh),
                corr=[_ring(a) for a in dv])
    du = [dt / dx * d for d in div]
    r = [u + d for u, d in zip(U, du)]
    D, phi = math.exp(-q), -math.expm1(-q) / q
    em1, em2 = -math.expm1(-q), -math.expm1(-2 * q)
    A, C, W = 0.5 * em2, em1 * em1 / q, (q - 2 * em1 + 0.5 * em2) / (q * q)
    ro, rn = U[0].clamp(min=SMALLR), r[0].clamp(min=SMALLR)
    w = [U[1 + c] / ro for c in range(3)]
    dw = [r[1 + c] / rn - w[c] for c in range(3)]
    out = list(r)
    out[0] = rn
    for c in range(3):
        out[1 + c] = rn * (D * w[c] + phi * dw[c])
    work_ = rn * sum(A * w[c] ** 2 + C * w[c] * dw[c] + W * dw[c] ** 2 for c in range(3))
    floor = 0.5 * (out[1] ** 2 + out[2] ** 2 + out[3] ** 2) / rn + 0.5 * (r[5] ** 2 + r[6] ** 2 + r[7] ** 2)
    out[4] = torch.maximum(r[4] - work_, floor)
    out[8] = r[8] * decay
    return torch.stack(out), du[0]


def _backtrace(fr, U, dtdx):
    """Trilinear samples of the fractions where each cell's gas came from."""
    n = U.shape[1]
    i = torch.arange(n, device=U.device, dtype=U.dtype)
    pos = [(i.view(1, 1, n), i.view(1, n, 1), i.view(n, 1, 1))[d] - dtdx * U[1 + d] / U[0] for d in range(3)]
    base = [p.floor() for p in pos]
    f = [p - b for p, b in zip(pos, base)]
    b = [(a.long() % n, (a.long() + 1) % n) for a in base]
    out = []
    for a in fr:
        a = a.reshape(-1)
        s = 0.0
        for c in range(8):
            h = (c & 1, c >> 1 & 1, c >> 2)
            wgt = 1.0
            for d in range(3):
                wgt = wgt * (f[d] if h[d] else 1 - f[d])
            s = s + wgt * a[(b[2][h[2]] * n + b[1][h[1]]) * n + b[0][h[0]]]
        out.append(s)
    return out


def _train(case, seed):
    """The trained weights and losses: Adam on the trainer's hashed mini-batches."""
    X, Y, _ = _pairs(case, seed)
    X, Y = torch.from_numpy(X).double().to(DEV), torch.from_numpy(Y).double().to(DEV)
    w = torch.from_numpy(_part_trained(seed)).double().to(DEV)
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    mask = (1 << 64) - 1
    losses = []
    for t in range(1, case["steps"] + 1):
        key = (seed * 0xD1B54A32D192ED03 + t * 0x9E3779B97F4A7C15) & mask
        with np.errstate(over="ignore"):
            z = np.uint64(key) + np.arange(case["batch"], dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z = z ^ (z >> np.uint64(31))
        i = torch.from_numpy((z % np.uint64(len(X))).astype(np.int64)).to(DEV)
        loss, g = _gradient(w, X[i], Y[i])
        losses.append(loss)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        w = w - case["lr"] * (m / (1 - 0.9 ** t)) / ((v / (1 - 0.999 ** t)).sqrt() + 1e-8)
    return dict(weights=w.cpu().numpy(), losses=np.array(losses))


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _train(case, seed)
    if kind == "ensemble":
        edges = [32] * case["n32"] + [64] * case["n64"] + [128] * case["n128"]
        out = []
        for c in _some(edges):
            n = edges[c]
            U = _initial(case, (n, n, n), seed * 1009 + c).double()
            for _ in range(case["steps"]):
                U = _step(case, U, *_rule(U, 1.0 / n), 1.0 / n)
            out.append(U.reshape(9, -1))
        return out
    dx = 1.0 / case["nx"]
    U = _initial(case, _grid_of(case), seed)
    if kind == "ct":
        U, B = _faces(U, seed)
        U, B = U.double(), B.double()
        for _ in range(case["steps"]):
            U, B = _ct_step(case, U, B, _rule(U, dx)[0], dx)
        return dict(faces=B, fields=U)
    U = U.double()
    if kind == "coupled":
        _, gen = _generators(seed + 2)
        dv = [a.double() for a in _modes(_grid_of(case), gen, 4, -2.0, 0.01, 3)]
        rho = U[0].float()
        fr = [(rho * f).double() / U[0] for f in _fractions(_grid_of(case), seed)]
        dt, ch, _ = _rule(U, dx)
        U, drho = _coupled_step(case, U, dv, dt, ch, 0.99, 0.1, dx)
        s1, s2 = _backtrace(fr, U, dt / dx)
        s2 = s2.clamp(0, 1)
        return dict(fields=U, density_perturbation=drho, species1=U[0] * torch.minimum(s1.clamp(min=0), 1 - s2),
                    species2=U[0] * s2)
    net = None
    if kind == "surrogate":
        net = (torch.from_numpy(np.load(WEIGHTS)).double().to(DEV), case["thr"])
    for _ in range(case["steps"]):
        U = _step(case, U, *_rule(U, dx), dx, net=net)
    return U if kind == "into" else dict(fields=U)
