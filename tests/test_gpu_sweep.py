"""Binary64 Adams-Bashforth steps whose z fluxes and update are one kernel
(k_sweep_update, blocks without one-launch stencils) against the one-launch stencils
and their update: the operations and their order are the same, so states and the
fluxes a call leaves are equal bit for bit.  Sizes: x rows below, at and past the
64-lane tile; z runs of one face tile, of just the longest run (31 cells), of one
more cell, with tiles left over; few rows and many.  (A blast of a few cells runs
into NaN with some limiters, on both sides alike.)
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

SIZES = [(4, 4, 4), (64, 5, 3 + 4), (65, 4, 31), (63, 7, 32), (130, 4, 70), (5, 40, 63)]


@pytest.mark.parametrize("sheared,bc", [(False, "even"), (True, "periodic")])
@pytest.mark.parametrize("reconop", [1, 2, 3, 4])
@pytest.mark.parametrize("n", SIZES)
def test_sweep_equals_one_launch(n, reconop, sheared, bc, monkeypatch):
    A = [[1., .5, 0.], [0., 1., .2], [0., 0., 1.]] if sheared else None
    g = ics.Grid(*n, ng=4, A=A)
    st = ics.initial_state(g, "blast", 21, radius=.2, p_in=10., p_out=.1)
    out = []
    for fill in (None, "0"):   # 0: EMF runs stay long and every stencil has its launch
        if fill is not None:
            monkeypatch.setenv("MHD_EMF_FILL_THREADS", fill)
        for overlap in (True, False):
            s = gpu.Solver(gpu.make_params(*n, ng=4, reconop=reconop, stepop=1, bc=bc), g)
            s.set_overlap(overlap)
            s.upload(st)
            tau = s.initialize(1e-4)
            for m in (1, 3):
                tau, _ = s.step(m, tau)
            out.append((s.download(), s.flux_stress(compute=False), tau))
            s.close()
    a, fa, ta = out[0]
    for b, fb, tb in out[1:]:
        assert ta == tb or (np.isnan(ta) and np.isnan(tb))
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k
        for q in range(24):
            assert np.array_equal(fa[q], fb[q], equal_nan=True), q
