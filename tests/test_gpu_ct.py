"""Constrained transport, one thread a corner of the owned block: the last face of
each family past the cells, blocks whose corners fill their workgroups and that
leave some over, flat and long ones, alone (second stream) and in the launch it
shares with the cell update.
Trajectories against the oracle at 1e-12 as in test_gpu_parity.py.
"""
import numpy as np
import pytest

import pyoracle as po
from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

SIZES = [(4, 5, 6), (7, 15, 15), (127, 127, 4), (130, 126, 5), (4, 4100, 4)]


@pytest.mark.parametrize("overlap", [False, True])
@pytest.mark.parametrize("stepop", [1, 2, 3])
@pytest.mark.parametrize("n", SIZES)
def test_ct_planes(n, stepop, overlap):
    g = ics.Grid(*n, ng=4)
    st = ics.initial_state(g, "rough", seed=7)
    s = gpu.Solver(gpu.make_params(*n, reconop=1, stepop=stepop, bc="periodic"), g)
    o = po.Oracle(po.make_params(*n, reconop=1, stepop=stepop, bc="periodic"), g)
    s.set_overlap(overlap)
    s.upload(st)
    o.set_state(st)
    s.initialize(1e-5)
    o.initialize(1e-5)
    t0 = t1 = 1e-5
    for _ in range(2):
        t0, _ = s.step(1, t0 if stepop == 1 else 1e-5)
        t1, _ = o.step(1, t1 if stepop == 1 else 1e-5)
    a, b = s.download(), o.get_state()
    for k in ("rho", "p", "vx", "vy", "vz", "bi", "bj", "bk"):
        assert np.linalg.norm(a[k] - b[k]) <= 1e-12 * np.linalg.norm(b[k]), k
    s.close()
