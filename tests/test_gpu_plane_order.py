"""Mixed Adams-Bashforth steps on planes of more than 128 workgroups, where the
predictor deals each plane to the XCDs in eighths: a periodic state repeated along
x and y evolves as one copy of it does on a block of small planes (which keeps the
fixed runs).  Both round in binary32 (6e-8) with face speeds of at most a cell a
step, so ten steps of a smooth flow agree within 1e-5 of each field's scale; the
state itself moves by 1e-2 a step, which a place left out or done twice shows.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

CELLS, FACES = ("rho", "vx", "vy", "vz", "p"), ("bi", "bj", "bk")
NG = 4


def repeat(a, n, reps):
    """interior of `a` (block n) repeated reps times along x and y, ghosts periodic"""
    idx = []
    for ax in range(3):
        extra = a.shape[ax] - (n[ax] + 2 * NG)      # 1 for the face family's axis
        m = n[ax] * reps[ax] + 2 * NG + extra
        idx.append((np.arange(m) - NG) % n[ax] + NG)
    return np.asfortranarray(a[np.ix_(*idx)])


# plane workgroups of the repeated block: below and above 128, with and without
# places left over by the eighths
@pytest.mark.parametrize("n,reps", [((60, 57, 6), (3, 3, 1)), ((60, 60, 6), (3, 3, 1)), ((125, 16, 5), (4, 4, 1))])
def test_repeated_state(n, reps):
    g = ics.Grid(*n, ng=NG)
    base = ics.initial_state(g, "orszag_tang", noise=0.)
    out = []
    for r in ((1, 1, 1), reps):
        m = tuple(a * b for a, b in zip(n, r))
        gr = ics.Grid(*m, ng=NG, hi=tuple(float(b) for b in r))
        st = dict(base)
        for k in CELLS + FACES:
            st[k] = repeat(base[k], n, r)
        s = gpu.Solver(gpu.make_params(*m, ng=NG, reconop=1, stepop=1, bc="periodic", precision="mixed"), gr)
        s.upload(st)
        tau = s.initialize(1e-3)
        for _ in range(10):
            tau, _ = s.step(1, tau)
        out.append(s.download())
        s.close()
    one, many = out
    for names in (("rho",), ("p",), ("vx", "vy", "vz"), FACES):
        scale = max(np.abs(one[k]).max() for k in names)
        for k in names:
            d = np.abs(many[k] - repeat(one[k], n, reps)).max()
            assert d <= 1e-5 * scale, (k, d / scale)
