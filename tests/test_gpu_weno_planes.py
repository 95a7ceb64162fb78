"""The binary64 WENO EMF with as few planes of scratch as it can do with (a block that
leaves the GPU no memory for more gets them): one plane of edges a slab, two, and
one more than half of the block's.  The slabs do not change the operations, so the
EMF equals that of one slab bit for bit, and a step's state too.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

N, NG = (20, 14, 9), 3


@pytest.mark.parametrize("sheared", [False, True])
@pytest.mark.parametrize("recon,eps", [(3, 1e-8), (4, 1e-8), (3, 1e-150)])
def test_few_planes(recon, eps, sheared, monkeypatch):
    A = [[1., .5, 0.], [0., 1., .2], [0., 0., 1.]] if sheared else None
    g = ics.Grid(*N, ng=NG, A=A)
    st = ics.initial_state(g, "blast" if sheared else "rough", seed=4)
    out = []
    for planes in (None, 0, 6, 7, 11):
        if planes is not None:
            monkeypatch.setenv("MHD_WENO_PLANES", str(planes))
        p = gpu.make_params(*N, ng=NG, reconop=recon, stepop=2, bc="periodic")
        p.eps = eps
        s = gpu.Solver(p, g)
        s.upload(st)
        s.initialize(1e-5)
        e = s.eijk()
        s.step(1, 1e-5)
        out.append((e, s.download()))
        s.close()
    for e, x in out[1:]:
        for a, b in ((e, out[0][0]), (x, out[0][1])):
            for k in b:
                assert np.isfinite(b[k]).all() and np.array_equal(a[k], b[k]), k
