"""The one-launch stencils of small blocks (k_stencils) against the oracle at the
sizes where their parts can go wrong: the smallest block, rows shorter and
longer than a 64-lane tile, a run axis just as long as a run (so that the last
run starts early), ej's column rows straddling workgroups (249 columns each), and
binary64 PDM on both sides of the rule that takes runs of 4 edges (256
workgroups in all).  EMFs are the oracle's bit for bit (the same operations in
the same order); fluxes carry erfc and exp, 1e-13 of each array's norm as in
test_gpu_parity.py.
"""
import numpy as np
import pytest

import pyoracle as po
from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

SIZES = [(4, 4, 4), (4, 5, 30), (5, 30, 4), (29, 23, 27), (70, 9, 33), (257, 6, 5)]


@pytest.mark.parametrize("reconop", [1, 2, 3, 4])
@pytest.mark.parametrize("n", SIZES)
def test_stencils_match_oracle(n, reconop):
    g = ics.Grid(*n, ng=4)
    st = ics.initial_state(g, "rough", seed=3)
    s = gpu.Solver(gpu.make_params(*n, reconop=reconop, stepop=2, bc="periodic"), g)
    o = po.Oracle(po.make_params(*n, reconop=reconop, stepop=2, bc="periodic"), g)
    s.upload(st)
    o.set_state(st)
    s.initialize(1e-4)
    o.initialize(1e-4)
    ref = o.ops()
    e = s.eijk()
    for k in ("ei", "ej", "ek"):
        assert np.array_equal(e[k], ref[k]), k
    for q, f in enumerate(s.flux_stress()):
        assert np.linalg.norm(f - ref["flux"][q]) <= 1e-13 * np.linalg.norm(ref["flux"][q]), q
    # the step forms both in one launch: the same arrays
    s.step(1, 1e-4)
    o.step(1, 1e-4)
    a, b = s.download(), o.get_state()
    for k in ("rho", "p", "vx", "vy", "vz", "bi", "bj", "bk"):
        assert np.linalg.norm(a[k] - b[k]) <= 1e-12 * np.linalg.norm(b[k]), k
    s.close()
