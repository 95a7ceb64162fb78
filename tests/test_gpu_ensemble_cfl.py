"""The CFL step that ensemble steps leave with a member, whatever ran on the member
between them: the minimum goes over every workgroup's partial, so a box whose CFL
limit is one hot cell returns what the same box stepped alone returns, bit for bit,
for hot cells in the workgroups that the pass over cells and boundary faces places
past the number of workgroups the cells alone would need.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

N, NG, TAU = 16, 3, 1e-4
NX = N + 2 * NG
# workgroups (256 cells) of the 48 that such a block has and that come after the
# cells' 42 in launch order; a cell near the middle of each that the block owns
GROUPS = (17, 23, 29, 35)


def hot_cell(w):
    for q in range(w * 256 + 128, w * 256 + 256):
        x = np.unravel_index(q, (NX, NX, NX))[::-1]
        if all(NG <= v < NG + N for v in x):
            return x
    raise AssertionError(w)


def box(place, precision):
    g = ics.Grid(N, N, N, ng=NG)
    st = ics.initial_state(g, "rough", seed=2)
    st["p"] = np.asfortranarray(st["p"].copy())
    st["p"][place] = 400.
    s = gpu.Solver(gpu.make_params(N, N, N, ng=NG, reconop=2, stepop=2, bc="periodic", precision=precision), g)
    s.upload(st)
    s.initialize(TAU)
    return s


def between_nothing(s):
    pass


def between_bxyz(s):
    s.bxyz()


def between_dt(s):
    s.eijk()          # leaves no partials: get_dt forms its own
    s.get_dt()


BETWEEN = {"nothing": between_nothing, "bxyz": between_bxyz, "dt": between_dt}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("between", sorted(BETWEEN))
@pytest.mark.parametrize("w", GROUPS)
def test_cfl_of_members(w, between, precision):
    s, o = box(hot_cell(w), precision), box(hot_cell(w), precision)
    free = o.get_dt()
    BETWEEN[between](s)
    with gpu.Ensemble([s], [TAU]) as e:
        for k in (3, 1, 2):
            e.step(k)
            _, cfl = o.step(k, TAU)
            assert s.step(0, TAU) == (TAU, cfl)
            assert s.get_dt() == o.get_dt()
            BETWEEN[between](s)
    cold = box((0, 0, 0), precision)   # a ghost cell, which the fill replaces
    assert free < .5 * cold.get_dt()   # the hot cell is the limit
    for c in (s, o, cold):
        c.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_recording_runs_nothing(precision):
    """making an ensemble records the steps and does not run them: a member whose state
    was uploaded since its last step forms its CFL step from that state"""
    s, o = box(hot_cell(GROUPS[0]), precision), box(hot_cell(GROUPS[1]), precision)
    st = o.download()
    s.upload(st)
    with gpu.Ensemble([s], [TAU]):
        assert s.get_dt() == o.get_dt()
    s.close()
    o.close()
