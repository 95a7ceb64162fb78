"""Where a call's returned step is left: more contexts alive than result slots, closed
and made again in between, each get their own step back.
"""
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu


def test_more_contexts_than_slots():
    n = (4, 4, 4)
    g = ics.Grid(*n, ng=4)
    st = ics.initial_state(g, "rough", seed=3)

    def make(tau):
        s = gpu.Solver(gpu.make_params(*n, reconop=2, stepop=2, bc="periodic"), g)
        s.upload(st)
        s.initialize(tau)
        return s

    taus = [1e-6 * (1 + q) for q in range(131)]
    alive = [make(t) for t in taus]
    cfl = alive[0].get_dt()
    for q in (0, 64, 127, 128, 130):
        alive[q].close()
        alive[q] = make(taus[q])
    assert all(s.get_dt() == cfl for s in alive)
    assert [s.step(1, t)[0] for s, t in zip(alive, taus)] == taus
    for s in alive:
        s.close()
