"""Workloads whose speed counts: what a program that uses this package runs.

Four kinds of case, each through the package's public entry points:

  step      ``Solver.step``: one block advanced by ``nsteps`` steps, over the
            reconstructions, steppers, precisions, boundaries and metrics
  ensemble  ``Ensemble.step``: independent boxes advanced together
  chain     the same Runge-Kutta step, routine by routine, as a driver that
            keeps its own time loop calls it
  train     one epoch of the learned reconstruction's training

``exact`` repeats a step, chain, ensemble or training in 64 bits with plain
torch from the scheme's formulas (tensor-product and affine grids).
Arrays are held as torch tensors of shape (nz, ny, nx): the library's
column-major (nx, ny, nz) arrays seen from the other end.
"""
import functools
import math
import random

import numpy as np
import torch

from mhd3d_mpi_fortran_amd import gpu, ics, shell
from mhd3d_mpi_fortran_amd import surrogate as sg

GAM, CFL, PDMB, EPS, ALPHA, BETA = 5. / 3., .3, 4., 1e-8, 2., 4.   # the deck's defaults
RECON = {"pdm": 1, "tvd": 2, "weno5": 3, "mpweno5": 4}
GHOSTS = {"pdm": 4, "tvd": 2, "weno5": 3, "mpweno5": 3}
STEPPER = {"ab2": 1, "rk2": 2, "rk3": 3}
NSTAGE = {"ab2": 1, "rk2": 2, "rk3": 3}
SHEAR = [[1., .5, 0.], [0., 1., 0.], [0., 0., 1.]]
STATE = ("rho", "vx", "vy", "vz", "p", "bi", "bj", "bk")
SLOT = {"rho": 0, "vx": 1, "vy": 2, "vz": 3, "p": 4, "bi": 8, "bj": 9, "bk": 10}
FACE = {"bi": 0, "bj": 1, "bk": 2}   # the axis a face array is normal to
DEV = "cuda"


# ---------------------------------------------------------------- the cases
def _step(name, n, recon, stepper, precision, bc="periodic", ic="vortex", metric="none", ng=4, nsteps=1, learned=False):
    return dict(name=name, kind="step", nx=n[0], ny=n[1], nz=n[2], recon=recon, stepper=stepper, precision=precision,
                bc=bc, ic=ic, metric=metric, ng=ng, nsteps=nsteps, learned=learned)


def listed():
    return [
        # the deck's default block, one call a step as the Fortran driver's time loop makes it: launches count
        _step("deck16", (16, 16, 16), "pdm", "rk2", "fp64", bc="even"),
        # a small ragged block, the most expensive limiter and stepper, reflecting walls
        _step("ragged-mpweno5", (37, 53, 29), "mpweno5", "rk3", "fp64", bc="even", ng=3, nsteps=4),
        # the 64^3 vortex in binary64, several steps between two looks at the state
        _step("vortex64", (64, 64, 64), "pdm", "rk2", "fp64", nsteps=5),
        # the same step routine by routine, as a driver that keeps the reference's call sequence
        dict(name="chain96", kind="chain", nx=96, ny=96, nz=96, recon="pdm", stepper="rk2", precision="mixed",
             bc="periodic", ic="vortex", metric="none", ng=4, nsteps=1, learned=False),
        # a batch of boxes of several sizes, stepped together
        dict(name="boxes8", kind="ensemble", sizes="32,96,64,48,32,64,96,48", recon="tvd", stepper="rk2",
             precision="mixed", bc="periodic", ic="blobs", metric="none", ng=3, nsteps=4, learned=False),
        # the spherical shell (general metric) in both precisions
        _step("shell-mixed", (96, 64, 128), "weno5", "rk2", "mixed", bc="shell", ic="dipole", metric="shell", ng=3,
              nsteps=2),
        _step("shell-fp64", (96, 64, 128), "weno5", "rk2", "fp64", bc="shell", ic="dipole", metric="shell", ng=3),
        # a ragged block of ordinary size with walls, Adams-Bashforth and TVD in fp32 stencils
        _step("ragged-tvd-ab2", (161, 117, 95), "tvd", "ab2", "mixed", bc="even", ic="blobs", ng=2, nsteps=2),
        # the sheared-box blast wave at full size: fp32 stencils, binary64, learned reconstruction
        _step("blast256-mixed", (256, 256, 256), "pdm", "ab2", "mixed", ic="blast", metric="shear"),
        _step("blast256-fp64", (256, 256, 256), "pdm", "ab2", "fp64", ic="blast", metric="shear"),
        _step("blast256-learned", (256, 256, 256), "pdm", "ab2", "mixed", ic="blast", metric="shear", learned=True),
        # training the learned reconstruction: one epoch over collected samples
        dict(name="train", kind="train", samples=131072, batch=1024, lr=5e-3),
    ]


# relative cost of a zone-stage, for the cap on drawn sizes
_COST = {"pdm": 1., "tvd": 1., "weno5": 5., "mpweno5": 8.}


def _sizes(rng, lo, hi, cap):
    """three extents around a size spread over its logarithm, at most `cap` zones"""
    while True:
        b = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        n = [max(8, int(round(b * rng.uniform(.6, 1.6)))) for _ in range(3)]
        if n[0] * n[1] * n[2] <= cap:
            return n


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["chain", "ensemble", "train"])
    if kind == "train":
        batch = rng.choice([256, 512, 1000, 1024, 2048])
        return dict(kind=kind, samples=batch * rng.randrange(20, 140) + rng.randrange(batch), batch=batch,
                    lr=rng.choice([1e-3, 5e-3]))
    recon = rng.choice(["pdm", "pdm", "tvd", "weno5", "mpweno5"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "ensemble":
        boxes = [rng.choice([24, 32, 37, 48, 64, 75, 96]) for _ in range(rng.randrange(2, 9))]
        while sum(n ** 3 for n in boxes) * _COST[recon] > 4e6:
            boxes[boxes.index(max(boxes))] = rng.randrange(17, 33)
        return dict(kind=kind, sizes=",".join(map(str, boxes)), recon=recon, stepper=rng.choice(["rk2", "rk3"]),
                    precision=precision, bc=rng.choice(["periodic", "even"]), ic=rng.choice(["vortex", "blobs"]),
                    metric="none", ng=rng.choice([GHOSTS[recon], 4]), nsteps=rng.randrange(1, 4), learned=False)
    stepper = rng.choice(["ab2", "rk2", "rk3"] if kind == "step" else ["rk2", "rk3"])
    metric = rng.choice(["none", "none", "shear"])
    learned = kind == "step" and recon == "pdm" and precision == "mixed" and rng.random() < .25
    n = _sizes(rng, 12, 240, 1.4e7 / (_COST[recon] * NSTAGE[stepper]))
    zones = n[0] * n[1] * n[2]
    most = int(1.4e7 / (_COST[recon] * NSTAGE[stepper] * zones))
    return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], recon=recon, stepper=stepper, precision=precision,
                bc="periodic" if metric == "shear" else rng.choice(["periodic", "even"]),
                ic="blast" if metric == "shear" else rng.choice(["vortex", "blast", "blobs"]), metric=metric,
                ng=rng.choice([GHOSTS[recon], 4]), nsteps=max(1, min(most, rng.choice([1, 1, 2, 5]))), learned=learned)


def work(case):
    """bytes: the state (8 binary64 words a zone) read and written once a
    step -- Adams-Bashforth also reads the previous one -- or the samples
    read once; flops: the reconstructions, moments and corner velocities of
    one zone's 3 faces and 3 edges per stage, or the net's forward and
    backward passes"""
    if case["kind"] == "train":
        n = case["samples"] // case["batch"] * case["batch"]
        return {"bytes": n * 56 * 4., "flops": n * 6. * (40 * 32 + 32 * 32 + 32 * 16)}
    if case["kind"] == "ensemble":
        zones = sum(int(n) ** 3 for n in case["sizes"].split(","))
    else:
        zones = case["nx"] * case["ny"] * case["nz"]
    words = 24 if case["stepper"] == "ab2" else 16
    per = {"pdm": 1700., "tvd": 900., "weno5": 8000., "mpweno5": 12000.}[case["recon"]]
    return {"bytes": zones * 8. * words * case["nsteps"], "flops": zones * per * NSTAGE[case["stepper"]] * case["nsteps"]}


# ------------------------------------------------------------ initial states
def _axis(t, d):
    """tensor of one axis' values, broadcastable over (nz, ny, nx)"""
    shape = [1, 1, 1]
    shape[2 - d] = -1
    return t.reshape(shape)


def _random(shape, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.rand(shape, generator=g, dtype=torch.float64, device=DEV)


def _initial(case, n, seed):
    """ghost-inclusive state of a tensor-product or sheared grid (ghosts zero)"""
    ng, rng = case["ng"], random.Random(seed)
    tot = [m + 2 * ng for m in n]
    ph = [rng.uniform(0., 2. * math.pi) for _ in range(12)]
    cen = [((torch.arange(tot[d], dtype=torch.float64, device=DEV) - ng + .5) / n[d]) for d in range(3)]
    X, Y, Z = (_axis(cen[d], d) for d in range(3))
    cs = (tot[2], tot[1], tot[0])
    one = torch.ones(cs, dtype=torch.float64, device=DEV)
    # the vortex carries 1e-3 of density noise; the others start smooth, as their resting states do
    noise = 2. * _random(cs, seed) - 1. if case["ic"] == "vortex" else 0. * one
    tp = 2. * math.pi
    # a smooth three-dimensional flow and field under the vortex and the blobs,
    # rest and a uniform field under the blast; each face family's component
    # depends on the transverse coordinates only, so the field starts free of
    # divergence
    if case["ic"] == "vortex":
        amp, rho0, p0, b0, bu = 1., 25. / (36. * math.pi), 5. / (12. * math.pi), 1. / math.sqrt(4. * math.pi), .05
    elif case["ic"] == "blast":
        amp, rho0, p0, b0, bu = 0., 1., .1, 0., .6
    else:
        amp, rho0, p0, b0, bu = .2, 1., 1., .05, .29
    st = dict(rho=rho0 * (1. + 1e-3 * noise), p=p0 * one,
              vx=-amp * torch.sin(tp * Y + ph[0]) + .1 * amp * torch.sin(tp * Z + ph[1]) + 0. * one,
              vy=amp * torch.sin(tp * X + ph[2]) + .1 * amp * torch.cos(tp * Z + ph[3]) + 0. * one,
              vz=.2 * amp * torch.sin(tp * Z + ph[4]) + .1 * amp * torch.cos(tp * X + ph[5]) + 0. * one)
    if case["ic"] == "blast":   # four hot spheres, nearest periodic image
        A = SHEAR if case["metric"] == "shear" else np.eye(3)
        hot = torch.zeros(cs, dtype=torch.bool, device=DEV)
        for _ in range(4):
            c = [rng.random() for _ in range(3)]
            d = [q - cq - torch.round(q - cq) for q, cq in zip((X, Y, Z), c)]
            e = [A[r][0] * d[0] + A[r][1] * d[1] + A[r][2] * d[2] for r in range(3)]
            hot |= (e[0] ** 2 + e[1] ** 2 + e[2] ** 2) < .1 ** 2
        st["p"] = torch.where(hot, 100. * one, st["p"])
    if case["ic"] == "blobs":   # three Gaussian blobs of density
        for _ in range(3):
            c, a, w = [rng.random() for _ in range(3)], rng.uniform(.5, 2.), rng.uniform(.05, .15)
            d = [q - cq - torch.round(q - cq) for q, cq in zip((X, Y, Z), c)]
            st["rho"] = st["rho"] + a * torch.exp(-(d[0] ** 2 + d[1] ** 2 + d[2] ** 2) / (w * w))
    for q, (key, d) in enumerate(FACE.items()):
        sh = list(cs)
        sh[2 - d] += 1
        t1, t2 = ((Y, Z), (Z, X), (X, Y))[d]
        st[key] = (b0 * (torch.sin(tp * t1 + ph[6 + q]) + .3 * torch.sin(2. * tp * t2 + ph[9 + q])) +
                   bu * (1., .9, .8)[d] + torch.zeros(sh, dtype=torch.float64, device=DEV))
    for key, a in st.items():
        own = [n[d] + (FACE.get(key) == d) for d in range(3)]
        z = torch.zeros_like(a)
        sl = tuple(slice(ng, ng + own[2 - t]) for t in range(3))
        z[sl] = a[sl]
        st[key] = z
    return st


@functools.lru_cache(maxsize=2)
def _shell_grid(nr, nth, nph, ng):
    g = shell.spherical_shell(nr, nth, nph, ng=ng)
    return g, shell.dipole_inflow(g, 0, noise=0.)


def _bc(case):
    return ("even", "even", "periodic") if case["bc"] == "shell" else case["bc"]


def _solver(case, n, seed):
    prm = gpu.make_params(n[0], n[1], n[2], ng=case["ng"], reconop=RECON[case["recon"]],
                          stepop=STEPPER[case["stepper"]], bc=_bc(case), precision=case["precision"],
                          surrogate=int(case["learned"]))
    if case["metric"] == "shell":
        g, st = _shell_grid(n[0], n[1], n[2], case["ng"])
        st = dict(st, rho=st["rho"] * (1. + .01 * (2. * _random((g.nz, g.ny, g.nx), seed).cpu().numpy().T - 1.)))
    else:
        g = ics.Grid(n[0], n[1], n[2], ng=case["ng"], A=SHEAR if case["metric"] == "shear" else None)
        st = {k: a.cpu().numpy().T for k, a in _initial(case, n, seed).items()}
    s = gpu.Solver(prm, g)
    s.upload(st)
    if case["learned"]:
        sg.set_weights(s, _net(seed))
        sg.configure(s, sg.THETA)
    tau = s.initialize(0. if case["stepper"] != "ab2" else 1e-4)
    return s, tau if case["stepper"] == "ab2" else .5 * s.get_dt()


def _net(seed):
    """weights of the net as training starts it"""
    g = torch.Generator().manual_seed(seed)
    w = []
    for rows, cols, scale in ((32, 40, 1.), (32, 32, 1.), (16, 32, .01)):
        w.append((2. * torch.rand(rows * cols, generator=g) - 1.) * scale / math.sqrt(cols))
        w.append(torch.zeros(rows))
    return torch.cat(w).numpy().astype(np.float32)


class _Held:
    """a device array of the library under the array interface torch reads"""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (ptr, False), "version": 2}


class _View:
    """the solver's device state as tensors, each of which keeps the solver
    (its memory's owner) alive; Adams-Bashforth rotates its buffers, so each
    address is looked up on every call"""

    def __init__(self, s):
        self.s, self.seen, self.lib = s, {}, gpu.lib()
        self.shape = {k: tuple(reversed(v)) for k, v in s._shapes().items()}

    def __call__(self):
        out = {}
        for k in STATE:
            ptr = self.lib.mhd_device_pointer(self.s.h, SLOT[k])
            t = self.seen.get((k, ptr))
            if t is None:
                t = self.seen[k, ptr] = torch.as_tensor(_Held(ptr, self.shape[k]), device=DEV)
                t.owner = self.s
            out[k] = t
        return out


# -------------------------------------------------------------------- cases
def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        s = gpu.Solver(gpu.make_params(16, 16, 16), ics.Grid(16, 16, 16))
        sg.load_samples(s, _samples(case, seed).float().cpu().numpy())
        return dict(kind=kind, s=s, case=case, seed=seed)
    if kind == "ensemble":
        members = []
        for b, n in enumerate(case["sizes"].split(",")):
            members.append(_solver(case, (int(n),) * 3, 1000 * seed + b))
        ens = gpu.Ensemble([s for s, _ in members], [t for _, t in members])
        return dict(kind=kind, ens=ens, views=[_View(s) for s, _ in members], nsteps=case["nsteps"])
    s, tau = _solver(case, (case["nx"], case["ny"], case["nz"]), seed)
    return dict(kind=kind, s=s, tau=tau, view=_View(s), nsteps=case["nsteps"], rk=case["stepper"] != "ab2",
                stages=NSTAGE[case["stepper"]])


def run(state):
    kind = state["kind"]
    if kind == "train":
        s, case = state["s"], state["case"]
        loss = sg.train(s, epochs=1, batch=case["batch"], lr=case["lr"], seed=state["seed"])
        return {"loss": loss, "weights": sg.get_weights(s)}
    if kind == "ensemble":
        state["ens"].step(state["nsteps"])
        return [v() for v in state["views"]]
    s = state["s"]
    if kind == "chain":
        L, h, tau = gpu.lib(), s.h, state["tau"]
        for _ in range(state["nsteps"]):
            tau_cfl = s.get_dt()
            s.set_tau(tau, tau)
            for stage in range(1, state["stages"] + 1):
                gpu._ck(L.mhd_eijk_lfm(h, gpu.STATE_CURRENT), "mhd_eijk_lfm")
                gpu._ck(L.mhd_flux_stress(h, gpu.STATE_CURRENT), "mhd_flux_stress")
                s.advance(stage)
                s.fill()
                s.bxyz()
    else:
        tau, tau_cfl = s.step(state["nsteps"], state["tau"])
    # the next call's step follows the CFL, as a driver's time loop does
    state["tau"] = .5 * tau_cfl if state["rk"] else tau
    return dict(state["view"](), tau=tau, tau_cfl=tau_cfl)


# ------------------------------------------------- the same in plain 64 bits
def _cut(a, d, lo, n):
    return a.narrow(2 - d, lo, n)


def _sgn(x):
    return torch.copysign(torch.ones_like(x), x)


def _fill(a, face, n, ng, bc):
    for d in range(3):
        f = 1 if face == d else 0
        own = n[d] + f
        idx = torch.arange(own + 2 * ng, device=a.device) - ng
        if bc == "periodic":
            idx = torch.where(idx < 0, idx + n[d], torch.where(idx >= own, idx - n[d], idx))
        elif f:
            idx = torch.where(idx < 0, -idx, torch.where(idx >= own, 2 * n[d] - idx, idx))
        else:
            idx = torch.where(idx < 0, -1 - idx, torch.where(idx >= own, 2 * n[d] - 1 - idx, idx))
        a = a.index_select(2 - d, idx + ng)
    return a


def _interp8(s):
    return (-3. * s[0] + 29. * s[1] - 139. * s[2] + 533. * s[3] + 533. * s[4] - 139. * s[5] + 29. * s[6] - 3. * s[7]) / 840.


def _pdm(fm2, fm1, f0, fp1, fi):
    fi = torch.maximum(torch.minimum(fm1, f0), torch.minimum(fi, torch.maximum(fm1, f0)))
    dm, d0, dp = PDMB * (fm1 - fm2), PDMB * (f0 - fm1), PDMB * (fp1 - f0)
    sm, s0, sp = _sgn(dm), _sgn(d0), _sgn(dp)
    fl = fi - s0 * torch.clamp((fi - fm1).abs() - (sm + s0).abs() * dm.abs(), min=0.)
    fr = fi + s0 * torch.clamp((f0 - fi).abs() - (s0 + sp).abs() * dp.abs(), min=0.)
    return fl, fr


def _tvd(fm2, fm1, f0, fp1, fi):
    a = (fm1 - fm2) / (f0 - fm1 + EPS)
    c = (f0 - fp1) / (fm1 - f0 + EPS)
    return (fm1 - (a + a.abs()) / (1. + a.abs()) * (fm1 - fi), f0 - (c + c.abs()) / (1. + c.abs()) * (f0 - fi))


def _weno(a, b, c, d, e):
    h = ((2. * a - 7. * b + 11. * c) / 6., (-b + 5. * c + 2. * d) / 6., (2. * c + 5. * d - e) / 6.)
    s = (13. / 12. * (a - 2. * b + c) ** 2 + .25 * (a - 4. * b + 3. * c) ** 2,
         13. / 12. * (b - 2. * c + d) ** 2 + .25 * (b - d) ** 2,
         13. / 12. * (c - 2. * d + e) ** 2 + .25 * (3. * c - 4. * d + e) ** 2)
    w = [g / (EPS + q) ** 2 for g, q in zip((.1, .6, .3), s)]
    t = w[0] + w[1] + w[2]
    return w[0] / t * h[0] + w[1] / t * h[1] + w[2] / t * h[2]


def _minmod(a, b):
    return .5 * (_sgn(a) + _sgn(b)) * torch.minimum(a.abs(), b.abs())


def _mp(u, a, b, c, d, e):
    h0, h1, h2 = a - 2. * b + c, b - 2. * c + d, c - 2. * d + e
    mr = _minmod(_minmod(4. * h1 - h2, 4. * h2 - h1), _minmod(h1, h2))
    ml = _minmod(_minmod(4. * h0 - h1, 4. * h1 - h0), _minmod(h0, h1))
    ul, md, lc = c + ALPHA * (c - b), .5 * (c + d - mr), .5 * (3. * c - b) + BETA * ml / 3.
    lo = torch.maximum(torch.minimum(torch.minimum(c, d), md), torch.minimum(torch.minimum(c, ul), lc))
    hi = torch.minimum(torch.maximum(torch.maximum(c, d), md), torch.maximum(torch.maximum(c, ul), lc))
    return u + _minmod(lo - u, hi - u)


_LO = {"pdm": -4, "tvd": -2, "weno5": -3, "mpweno5": -3}


def _limit(s, recon):
    """left and right states from the taps s of a face's stencil"""
    if recon == "pdm":
        return _pdm(s[2], s[3], s[4], s[5], _interp8(s))
    if recon == "tvd":
        return _tvd(s[0], s[1], s[2], s[3], .5 * (s[1] + s[2]))
    lt, rt = (s[0], s[1], s[2], s[3], s[4]), (s[5], s[4], s[3], s[2], s[1])
    wl, wr = _weno(*lt), _weno(*rt)
    return (_mp(wl, *lt), _mp(wr, *rt)) if recon == "mpweno5" else (wl, wr)


def _recon(a, d, n, ng, recon):
    """states at the n+1 owned faces along axis d"""
    lo = _LO[recon]
    return _limit([_cut(a, d, ng + m, n + 1) for m in range(lo, -lo)], recon)


def _moments(lam, v, side):
    a = torch.sqrt(lam)
    b = .5 * torch.exp(-lam * v * v) / (a * math.sqrt(math.pi))
    v0 = .5 * torch.special.erfc(-side * a * v)
    return v0, v * v0 + side * b


def _flux(q, d, nrm, n, ng, recon):
    """the 8 face products of the faces normal to axis d"""
    own = []
    for a in q:
        for t in range(3):
            if t != d:
                a = _cut(a, t, ng, n[t])
        own.append(_recon(a, d, n[d], ng, recon))
    out = [0.] * 8
    for side, pick in ((1., 0), (-1., 1)):
        r, u, v, w, p, x, y, z = (o[pick] for o in own)
        vel, b = (u, v, w), (x, y, z)
        un = nrm[0] * u + nrm[1] * v + nrm[2] * w
        bn = nrm[0] * x + nrm[1] * y + nrm[2] * z
        eng = .5 * r * (u * u + v * v + w * w) + p / (GAM - 1.)
        v0, v1 = _moments(r / (2. * p), un, side)
        out[0] = out[0] + r * v1
        for c in range(3):
            out[1 + c] = out[1 + c] + r * vel[c] * v1 + p * nrm[c] * v0
        out[4] = out[4] + (eng + .5 * p) * v1 + .5 * p * un * v0
        bsq = x * x + y * y + z * z
        v0, _ = _moments(r / (2. * p + bsq), un, side)
        for c in range(3):
            out[5 + c] = out[5 + c] + (.5 * bsq * nrm[c] - b[c] * bn) * v0
    return out


def _corner(v, d1, d2, n, ng, recon):
    """corner velocity of the edges along the third axis; cv(o1, o2): the cell
    at those offsets along d1 and d2 from the edge"""
    e = 3 - d1 - d2
    v = _cut(v, e, ng, n[e])

    def cv(o1, o2):
        return _cut(_cut(v, d1, ng + o1, n[d1] + 1), d2, ng + o2, n[d2] + 1)

    if recon == "pdm":
        line = _interp8([_cut(v, d1, ng + m, n[d1] + 1) for m in range(-4, 4)])
        vi = _interp8([_cut(line, d2, ng + m, n[d2] + 1) for m in range(-4, 4)])
        a00, a10 = _pdm(cv(-2, -1), cv(-1, -1), cv(0, -1), cv(1, -1), vi)
        b00, b01 = _pdm(cv(-1, -2), cv(-1, -1), cv(-1, 0), cv(-1, 1), vi)
        b10, b11 = _pdm(cv(0, -2), cv(0, -1), cv(0, 0), cv(0, 1), vi)
        a01, a11 = _pdm(cv(-2, 0), cv(-1, 0), cv(0, 0), cv(1, 0), vi)
    elif recon == "tvd":
        vi = .25 * (cv(-1, -1) + cv(0, -1) + cv(0, 0) + cv(-1, 0))
        a00, a10 = _tvd(cv(-2, 0), cv(-1, 0), cv(0, 0), cv(1, 0), vi)
        b00, b01 = _tvd(cv(0, -2), cv(0, -1), cv(0, 0), cv(0, 1), vi)
        b10, b11, a01, a11 = b00, b01, a00, a10
    else:
        def two(first, second):
            l, r = _limit([_cut(v, first, ng + m, n[first] + 1) for m in range(-3, 3)], recon)
            return [_limit([_cut(f, second, ng + m, n[second] + 1) for m in range(-3, 3)], recon) for f in (l, r)]

        (b00, b01), (b10, b11) = two(d1, d2)
        (a00, a01), (a10, a11) = two(d2, d1)

    def sel(p, q, r, c, va, vb):   # the direction of the larger difference
        s = _sgn((cv(*p) - cv(*c)).abs() - (cv(*q) - cv(*r)).abs())
        return torch.where(s > 0., va, vb)

    c00 = sel((-2, -1), (-1, -2), (-1, -1), (-1, -1), a00, b00)
    c10 = sel((1, -1), (0, -2), (0, -1), (0, -1), a10, b10)
    c01 = sel((-2, 0), (-1, 1), (-1, 0), (-1, 0), a01, b01)
    c11 = sel((1, 0), (0, 1), (0, 0), (0, 0), a11, b11)
    return .25 * (c00 + c01 + c10 + c11)


def _emf(w, b, vf, e, fac, n, ng, recon):
    """EMF of the edges along axis e from the face-normal velocities w"""
    d1, d2 = (e + 1) % 3, (e + 2) % 3
    v1, v2 = _corner(w[d1], d1, d2, n, ng, recon), _corner(w[d2], d1, d2, n, ng, recon)
    b1 = _cut(_cut(b[d1], e, ng, n[e]), d1, ng, n[d1] + 1)
    b2 = _cut(_cut(b[d2], e, ng, n[e]), d2, ng, n[d2] + 1)
    b1l, b1r = _recon(b1, d2, n[d2], ng, recon)
    b2l, b2r = _recon(b2, d1, n[d1], ng, recon)
    f = _cut(vf, e, ng, n[e])
    eta = .25 * sum(_cut(_cut(f, d1, ng + o, n[d1] + 1), d2, ng + m, n[d2] + 1) for o in (-1, 0) for m in (-1, 0))
    out = (-v1 * torch.where(_sgn(v1) > 0., b2l, b2r) + v2 * torch.where(_sgn(v2) > 0., b1l, b1r) +
           eta * (b1l + b2r - b1r - b2l))
    return out * fac


class _Exact:
    """one block of the scheme on a uniform or sheared periodic grid"""

    def __init__(self, case, n, seed):
        self.n, self.ng, self.recon, self.bc = n, case["ng"], case["recon"], case["bc"]
        A = np.array(SHEAR) if case["metric"] == "shear" else np.eye(3)
        C = np.array([np.cross(A[:, (d + 1) % 3], A[:, (d + 2) % 3]) for d in range(3)])
        ln, J = np.linalg.norm(C, axis=1), np.linalg.det(A)
        self.nrm = C / ln[:, None]
        self.h = [J / ln[d] / n[d] for d in range(3)]      # physical spacing of the face families
        self.dc = [1. / n[d] for d in range(3)]
        self.ct = 1. / ln
        self.ef = [ln[(d + 1) % 3] * ln[(d + 2) % 3] / J for d in range(3)]
        self.M = A * (ln / J)[None, :]
        st = _initial(case, n, seed)
        self.x = [st[k] for k in STATE]
        self.fill()

    def fill(self):
        self.x = [_fill(a, FACE.get(k), self.n, self.ng, self.bc) for k, a in zip(STATE, self.x)]

    def cell_b(self, x):
        m = [.5 * (_cut(x[5 + d], d, 0, x[0].shape[2 - d]) + _cut(x[5 + d], d, 1, x[0].shape[2 - d])) for d in range(3)]
        return [self.M[r, 0] * m[0] + self.M[r, 1] * m[1] + self.M[r, 2] * m[2] for r in range(3)]

    def dt(self):
        r, u, v, w, p = self.x[:5]
        b = self.cell_b(self.x)
        fast = torch.sqrt(u * u + v * v + w * w) + torch.sqrt((b[0] ** 2 + b[1] ** 2 + b[2] ** 2 + GAM * p) / r)
        return float((CFL / (fast * sum(1. / h for h in self.h))).min())

    def products(self, x):
        """face fluxes and edge EMFs of the state x"""
        b = self.cell_b(x)
        F = [_flux(x[:5] + b, d, self.nrm[d], self.n, self.ng, self.recon) for d in range(3)]
        r, u, v, w = x[:4]
        vf = torch.sqrt(u * u + v * v + w * w) + torch.sqrt((b[0] ** 2 + b[1] ** 2 + b[2] ** 2) / r)
        wn = [m[0] * u + m[1] * v + m[2] * w for m in self.nrm]
        E = [_emf(wn, x[5:], vf, e, self.ef[e], self.n, self.ng, self.recon) for e in range(3)]
        return F, E

    def own(self, a, key):
        for d in range(3):
            a = _cut(a, d, self.ng, self.n[d] + (FACE.get(key) == d))
        return a

    def advance(self, FE, tau, mix=None, prev=None):
        """the current state's update; mix = (weight of prev, weight, divisor)"""
        F, E = FE
        n = self.n
        c = [self.own(a, k) for k, a in zip(STATE, self.x)]

        def div(q):
            return sum((_cut(F[d][q], d, 1, n[d]) - _cut(F[d][q], d, 0, n[d])) / self.h[d] for d in range(3))

        def comb(new, old):
            return new if mix is None else (mix[0] * old + mix[1] * new) / mix[2]

        U = self.conserved(c)
        P = self.conserved(prev) if prev is not None else [None] * 5
        rho = comb(U[0] - tau * div(0), P[0])
        m = [U[1 + q] - tau * div(1 + q) for q in range(3)]
        eng = comb(U[4] - tau * div(4), P[4])
        hm = [comb(m[q], P[1 + q]) for q in range(3)]
        p = (GAM - 1.) * (eng - .5 * (hm[0] ** 2 + hm[1] ** 2 + hm[2] ** 2) / rho)
        vel = [comb(m[q] - tau * div(5 + q), P[1 + q]) / rho for q in range(3)]
        faces = []
        for d in range(3):
            a, b = (d + 1) % 3, (d + 2) % 3
            curl = ((_cut(E[b], a, 1, n[a]) - _cut(E[b], a, 0, n[a])) / self.dc[a] -
                    (_cut(E[a], b, 1, n[b]) - _cut(E[a], b, 0, n[b])) / self.dc[b])
            faces.append(comb(c[5 + d] - tau * self.ct[d] * curl, prev[5 + d] if prev is not None else None))
        new = [rho] + vel + [p] + faces
        ng, out = self.ng, []
        for k, a, o in zip(STATE, self.x, new):
            z = a.clone()
            z[tuple(slice(ng, ng + q) for q in o.shape)] = o
            out.append(z)
        self.x = out
        self.fill()

    @staticmethod
    def conserved(c):
        r, u, v, w, p = c[:5]
        return [r, r * u, r * v, r * w, .5 * r * (u * u + v * v + w * w) + p / (GAM - 1.)]

    def rk(self, nst, tau):
        prev = [self.own(a, k) for k, a in zip(STATE, self.x)]
        mixes = [None, (1., 1., 2.)] if nst == 2 else [None, (3., 1., 4.), (1., 2., 3.)]
        for mix in mixes:
            self.advance(self.products(self.x), tau, mix, prev if mix else None)

    def outputs(self):
        return dict(zip(STATE, self.x))


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if case["metric"] == "shell" or case["learned"]:
        return None   # curved cells and the net's 16-bit products: no plain counterpart here
    if kind == "ensemble":
        out = []
        for b, n in enumerate(case["sizes"].split(",")):
            x = _Exact(case, (int(n),) * 3, 1000 * seed + b)
            tau = .5 * x.dt()
            for _ in range(case["nsteps"]):
                x.rk(NSTAGE[case["stepper"]], tau)
            out.append(x.outputs())
        return out
    x = _Exact(case, (case["nx"], case["ny"], case["nz"]), seed)
    tau = .5 * x.dt()
    if case["stepper"] != "ab2":
        for _ in range(case["nsteps"]):
            cfl = x.dt()
            x.rk(NSTAGE[case["stepper"]], tau)
    else:
        tau0, old = 3e-4, x.x   # the reference's hard-coded first step
        for _ in range(case["nsteps"]):
            cfl = tau = x.dt()
            c = .5 * tau / tau0
            half = [a + c * (a - b) for a, b in zip(x.x, old)]
            tau0, old = tau, x.x
            x.advance(x.products(half), tau)
    return dict(x.outputs(), tau=tau, tau_cfl=cfl)


# ------------------------------------------------------------------ training
def _samples(case, seed):
    """face samples as collection gives them: normalised 5-point windows of 8
    variables, smooth with a kink here and there, and PDM's face states"""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n = case["samples"]

    def rnd(*shape):
        return torch.rand(shape, generator=g, dtype=torch.float64, device=DEV)

    j = torch.arange(8, dtype=torch.float64, device=DEV) - 3.5
    k, ph, sl, kink, at = rnd(n, 8, 1), rnd(n, 8, 1), 2. * rnd(n, 8, 1) - 1., rnd(n, 8, 1), 4. * rnd(n, 8, 1) - 2.
    f = torch.sin(.6 * k * j + 6.3 * ph) + sl * j + .3 * (kink > .8) * (j - at).abs()
    w = f[:, :, 2:7]
    c = .5 * (w[:, :, 1:2] + w[:, :, 2:3])
    s = (w - c).abs().amax(dim=2, keepdim=True) + 1e-3
    s8 = [f[:, :, m] for m in range(8)]
    fl, fr = _limit(s8, "pdm")
    x = ((w - c) / s).reshape(n, 40)
    y = torch.cat([(q - c[:, :, 0]) / s[:, :, 0] for q in (fl, fr)], dim=1)
    return torch.cat([x, y], dim=1)


def _exact_train(case, seed):
    """one epoch of Adam in 64 bits on the CPU: the net's deterministic start, one
    permutation of the samples, cosine decay"""
    mask = (1 << 64) - 1
    z = [(0x9E3779B97F4A7C15 * (seed + 1)) & mask]

    def uniform():
        z[0] = (z[0] + 0x9E3779B97F4A7C15) & mask
        r = z[0]
        r = ((r ^ (r >> 30)) * 0xBF58476D1CE4E5B9) & mask
        r = ((r ^ (r >> 27)) * 0x94D049BB133111EB) & mask
        return float((r ^ (r >> 31)) >> 11) / 9007199254740992.

    par = []
    for rows, cols, scale in ((32, 40, 1.), (32, 32, 1.), (16, 32, float(np.float32(.01)))):
        a = 1. / math.sqrt(cols)
        w = torch.tensor([(2. * uniform() - 1.) * a for _ in range(rows * cols)]).double().float().double() * scale
        par += [w.float().double().reshape(rows, cols), torch.zeros(rows, dtype=torch.float64)]
    par = [p.requires_grad_(True) for p in par]
    data = _samples(case, seed).float().double().cpu()
    n, batch = data.shape[0], case["batch"]
    m64 = (1 << 64) - 1
    q = (0xD1B54A32D192ED03 ^ (seed & 0xffffffff)) * 6364136223846793005 + 1442695040888963407 & m64
    mult = (q >> 17) % n | 1
    while math.gcd(mult, n) != 1:
        mult += 2
    first, nb, tot = (q >> 7) % n, n // batch, 0.
    mom, var = [torch.zeros_like(p) for p in par], [torch.zeros_like(p) for p in par]
    for b in range(nb):
        f = (first + b * batch * (mult % n)) % n
        s = data[torch.tensor([(f + i * mult) % n for i in range(batch)])]
        x, t = s[:, :40], s[:, 40:]
        x5 = x.reshape(-1, 8, 5)
        lin = (-x5[:, :, 0] + 7. * x5[:, :, 1] + 7. * x5[:, :, 2] - x5[:, :, 3]) / 12.
        gate = (x5[:, :, :-2] - 2. * x5[:, :, 1:-1] + x5[:, :, 2:]).abs().amax(dim=2)
        h = x
        for w, o in zip(par[0:4:2], par[1:4:2]):
            a = h @ w.T + o
            h = a * torch.sigmoid(1.702 * a)
        y = lin.repeat(1, 2) + gate.repeat(1, 2) * (h @ par[4].T + par[5])
        sq = ((y - t) ** 2).sum()
        tot += float(sq.detach())
        grads = torch.autograd.grad(sq / (batch * 16), par)
        lr = case["lr"] * .5 * (1. + math.cos(math.pi * b / nb))
        with torch.no_grad():
            for p, gr, mo, va in zip(par, grads, mom, var):
                mo.mul_(.9).add_(gr, alpha=.1)
                va.mul_(.999).addcmul_(gr, gr, value=.001)
                p -= lr * (mo / (1. - .9 ** (b + 1))) / ((va / (1. - .999 ** (b + 1))).sqrt() + 1e-8)
    return {"loss": tot / (nb * batch * 16),
            "weights": torch.cat([p.detach().reshape(-1) for p in par])}
