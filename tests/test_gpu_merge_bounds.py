"""Which binary64 blocks run a stage's stencils in one launch, and its update and CT in
one: those of a size, or so narrow, that this was the faster way by measurement.  CT
has launches of its own elsewhere.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu


# TVD below its bound of 2^22 cells and from there on; the others are past it
@pytest.mark.parametrize("reconop,n,merged", [
    (2, (128, 128, 128), True), (2, (161, 161, 161), True), (2, (162, 162, 162), False),
    (1, (162, 162, 162), True), (3, (162, 162, 162), True), (4, (162, 162, 162), True)])
def test_runge_kutta_blocks(reconop, n, merged):
    g = ics.Grid(*n, ng=4)
    s = gpu.Solver(gpu.make_params(*n, ng=4, reconop=reconop, stepop=2, bc="periodic"), g)
    s.upload(ics.initial_state(g, "orszag_tang"))
    s.initialize(1e-5)
    s.profile(True)
    s.step(1, 1e-5)
    ct, _ = s.profile_read("ct")
    s.close()
    assert ct == (0 if merged else 2)


# binary64 Adams-Bashforth blocks from 2^21 cells on: z fluxes and update in one kernel
# (two flux launches) where x fills 1/2 (PDM), 3/8 (TVD) or 3/4 (WENO) of its 64-lane
# tiles; narrower ones all fluxes by themselves (three), PDM all stencils at once (one)
@pytest.mark.parametrize("reconop,n,flux", [
    (1, (31, 270, 260), 1), (1, (32, 260, 260), 2), (1, (4, 800, 700), 1),
    (2, (23, 310, 300), 3), (2, (24, 300, 300), 2), (2, (65, 182, 180), 2),
    (3, (47, 220, 210), 3), (3, (48, 212, 212), 2), (4, (129, 130, 130), 3), (4, (64, 190, 190), 2)])
def test_adams_bashforth_rows(reconop, n, flux, monkeypatch):
    g = ics.Grid(*n, ng=4)
    st = ics.initial_state(g, "orszag_tang")
    out = []
    for fill in (None, "0"):   # 0: EMF runs stay long and nothing shares a launch with them
        if fill is not None:
            monkeypatch.setenv("MHD_EMF_FILL_THREADS", fill)
        s = gpu.Solver(gpu.make_params(*n, ng=4, reconop=reconop, stepop=1, bc="periodic"), g)
        s.upload(st)
        tau = s.initialize(1e-4)
        s.profile(True)
        tau, _ = s.step(1, tau)
        if fill is None:
            assert s.profile_read("flux")[0] == flux
        s.profile(False)
        s.step(2, tau)
        out.append((s.download(), s.flux_stress(compute=False)))
        s.close()
    (a, fa), (b, fb) = out
    for k in a:
        assert np.isfinite(a[k]).all() and np.array_equal(a[k], b[k]), k
    for q in range(24):
        assert np.array_equal(fa[q], fb[q]), q
