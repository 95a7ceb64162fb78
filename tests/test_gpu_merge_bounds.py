"""Which binary64 blocks run a stage's stencils in one launch, and its update and CT in
one: those of a size to which that was the faster way by measurement.  CT has
launches of its own elsewhere.
"""
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
