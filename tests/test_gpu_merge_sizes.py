"""Binary64 Runge-Kutta blocks from 2^21 cells on, which form a stage's stencils in one
launch, against a launch per direction (two streams): the same operations in the
same order, so the states are equal bit for bit.  Just at, and past, 2^21 cells.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reconop,stepop", [(1, 2), (2, 3), (3, 2), (4, 2)])
@pytest.mark.parametrize("n", [(128, 128, 128), (67, 250, 127)])
def test_one_launch_of_large_blocks(n, reconop, stepop, monkeypatch):
    g = ics.Grid(*n, ng=4)
    st = ics.initial_state(g, "orszag_tang")
    out = []
    for fill in (None, "0"):   # 0: a launch per direction
        if fill is not None:
            monkeypatch.setenv("MHD_EMF_FILL_THREADS", fill)
        s = gpu.Solver(gpu.make_params(*n, ng=4, reconop=reconop, stepop=stepop, bc="periodic"), g)
        if fill is not None:
            s.set_overlap(True)
        s.upload(st)
        s.initialize(1e-4)
        s.step(2, 1e-4)
        out.append(s.download())
        s.close()
    for k in out[0]:
        assert np.isfinite(out[0][k]).all() and np.array_equal(out[0][k], out[1][k]), k
