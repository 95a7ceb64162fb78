"""Divisions in binary64 at the ends of the number range.

The limiters divide by differences of the field plus eps.  Whatever eps and the
field's scale, a state that the oracle finds finite is finite, and reconstruct_3d
equals the oracle's bit for bit where the operations are the same: all of them for
eps below 2^-400, and for a larger eps as long as no quotient of the oracle's is
subnormal (fields from 2^-900 to 2^240).

Past that (2^252, 2^253: the oracle's WENO weights are subnormal before they are
normalised) eps is lost beside the smoothness indicators, so the field's power of two
passes through: the reconstruction is that of the field times 2^-50, to 4 places of
2^-52 of the stencil's largest candidate value (at most 11/3 of the field's largest)
for each of the three products of a weight that is one place off.
"""
import numpy as np
import pytest

import pyoracle as po
from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

N, NG = (20, 9, 7), 4
NX = tuple(n + 2 * NG for n in N)


def field(flats=True):
    f = np.random.default_rng(5).uniform(-1., 1., NX)
    if flats:
        f[:, ::3] = .25
        f[::5] *= 1e-6
        f[4:11, 2] = 0.
    return f


def run(recon, eps, f):
    p = gpu.make_params(*N, ng=NG, reconop=recon)
    p.eps = eps
    s = gpu.Solver(p, ics.Grid(*N, ng=NG))
    out = [gpu.reconstruct(s, f, (N[0] + 1, N[1], N[2]), 1), gpu.reconstruct(s, f, (N[0], N[1] + 1, N[2]), 2)]
    s.close()
    return [a for pair in out for a in pair]


def oracle(recon, eps, f):
    p = po.make_params(*N, ng=NG, reconop=recon)
    p.eps = eps
    out = [po.reconstruct(p, f, (N[0] + 1, N[1], N[2]), 1), po.reconstruct(p, f, (N[0], N[1] + 1, N[2]), 2)]
    return [a for pair in out for a in pair]


CASES = [(r, e, k) for r in (2, 3, 4) for e in (0., 1e-155, 7e-155, 1e-121, 1e-120, 1e-300, 1e-310, 5e-324, -1e-8)
         for k in (-900, -500, -254, -60, 0, 120, 240, 252, 255) if e < 2.**-400 or k <= 240]
CASES += [(2, e, k) for e in (0., 1e-310, 1e-8) for k in (-1070, -1040, -1020, 1000, 1021)]
CASES += [(r, e, k) for r in (1, 2, 3, 4) for e in (1e-8, 1e-20, 1e-100, 1.) for k in (-900, -500, -60, 0, 120, 240)]


@pytest.mark.parametrize("recon", [1, 2, 3, 4])
def test_reconstruction_over_the_range(recon):
    base = field()
    for r, eps, k in CASES:
        if r != recon:
            continue
        f = np.ldexp(base, k)
        with np.errstate(all="ignore"):
            ref = oracle(r, eps, f)
        for a, b in zip(run(r, eps, f), ref):
            assert np.array_equal(a, b, equal_nan=True), (eps, k)


@pytest.mark.parametrize("recon", [3, 4])
@pytest.mark.parametrize("k", [252, 253])
def test_weights_of_large_fields(recon, k):
    f = field(flats=False)
    small = run(recon, 1e-8, np.ldexp(f, k - 50))
    for a, b in zip(run(recon, 1e-8, np.ldexp(f, k)), small):
        assert np.isfinite(a).all()
        assert np.abs(np.ldexp(a, -k) - np.ldexp(b, 50 - k)).max() <= 3 * 4 * 2.**-52 * 11. / 3.


@pytest.mark.parametrize("rest", [False, True])
@pytest.mark.parametrize("sheared", [False, True])
@pytest.mark.parametrize("recon", [1, 2])
def test_flux_of_a_subnormal_pressure(recon, sheared, rest):
    """rho / 2p is finite and so are the fluxes (thermal speed 1e-153), of a gas at rest
    too; 1e-13 of each array's norm as in test_gpu_parity.py.  The sheared grid is
    A = I."""
    g = ics.Grid(*N, ng=NG, A=np.eye(3).tolist() if sheared else None)
    g0 = ics.Grid(*N, ng=NG)
    st = ics.initial_state(g0, "rough", seed=3)
    st["p"] = np.full_like(st["p"], 1e-310)
    st["rho"] = np.asfortranarray(1e-6 * st["rho"])
    if rest:
        for k in ("vx", "vy", "vz"):
            st[k] = np.zeros_like(st[k])
    s = gpu.Solver(gpu.make_params(*N, ng=NG, reconop=recon, stepop=2, bc="periodic"), g)
    o = po.Oracle(po.make_params(*N, ng=NG, reconop=recon, stepop=2, bc="periodic"), g0)
    s.upload(st)
    o.set_state(st)
    s.initialize(1e-9)
    o.initialize(1e-9)
    ref = o.ops()["flux"]
    for q, f in enumerate(s.flux_stress()):
        assert np.isfinite(ref[q]).all() and np.isfinite(f).all(), q
        assert np.linalg.norm(f - ref[q]) <= 1e-13 * np.linalg.norm(ref[q]), q
    s.close()


@pytest.mark.parametrize("eps,scale,flux", [(1e-8, 1., 2), (1e-8, 2.**450, 3), (1e-200, 1., 3)])
def test_sweep_needs_divisors_in_range(eps, scale, flux, monkeypatch):
    """the z sweep (two flux launches a step) divides by the spacings and by the
    limiters' differences in the short way; other blocks keep a launch per flux"""
    monkeypatch.setenv("MHD_EMF_FILL_THREADS", "0")
    n = (60, 6, 7)
    g = ics.Grid(*n, ng=NG, hi=(scale, scale, scale))
    p = gpu.make_params(*n, ng=NG, reconop=2, stepop=1, bc="periodic")
    p.eps = eps
    s = gpu.Solver(p, g)
    s.upload(ics.initial_state(ics.Grid(*n, ng=NG), "rough", seed=3))
    tau = s.initialize(1e-4)
    s.profile(True)
    s.step(1, tau)
    assert s.profile_read("flux")[0] == flux
    s.close()
