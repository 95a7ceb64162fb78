"""Cell B after mixed-precision Runge-Kutta steps, whose stages leave it out until the
last stage of a call: several steps of one call, the same steps a call each and
(periodic boxes) the members of an ensemble hold the same bx, by and bz, and
get_bxyz on that state forms them again, bit for bit.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

N, TAU = (9, 8, 11), 1e-4


def solver(stepop, sheared, bc):
    A = [[1., .5, 0.], [0., 1., .2], [0., 0., 1.]] if sheared else None
    g = ics.Grid(*N, ng=4, A=A)
    s = gpu.Solver(gpu.make_params(*N, ng=4, reconop=2, stepop=stepop, bc=bc, precision="mixed"), g)
    s.upload(ics.initial_state(g, "blast" if sheared else "rough", seed=3))
    s.initialize(TAU)
    return s


@pytest.mark.parametrize("sheared,bc", [(False, "periodic"), (False, "even"), (True, "periodic")])
@pytest.mark.parametrize("stepop", [2, 3])
def test_cellb_after_steps(stepop, sheared, bc):
    a, b, c = (solver(stepop, sheared, bc) for _ in range(3))
    a.step(3, TAU)
    for _ in range(3):
        b.step(1, TAU)
    e = gpu.Ensemble([c], [TAU])
    e.step(3)
    e.close()
    x = a.download()
    a.bxyz()
    for other in (a, b, c):
        y = other.download()
        for k in x:
            assert np.array_equal(x[k], y[k]), k
    for s in (a, b, c):
        s.close()
