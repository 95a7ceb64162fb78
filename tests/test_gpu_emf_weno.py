"""The binary64 WENO EMF (k_weno_lines, k_emf_weno), slab by slab.

Against the oracle the EMF is pinned bit for bit on small blocks
(test_gpu_parity.py), which one slab of the scratch holds.  Here a block whose
edge planes need several slabs is compared with two blocks of half its height
cut out of it, each of which one slab holds: every edge has the same stencil
values in both, so the results are the same bits wherever a slab ends.
"""
import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics

pytestmark = pytest.mark.gpu

NZ, NG = 40, 3
NX, NY = 180, 170
SCRATCH = 160 << 20    # kWenoScratch


def _eijk(nz, st, recon):
    g = ics.Grid(NX, NY, nz, ng=NG)
    s = gpu.Solver(gpu.make_params(NX, NY, nz, ng=NG, reconop=recon, stepop=2), g)
    s.upload(st)
    e = s.eijk()
    s.close()
    return e


@pytest.mark.parametrize("recon", [3, 4])
def test_slabs_equal_single_slab_blocks(recon):
    held = SCRATCH // (18 * 8 * (NX + 2 * NG) * (NY + 2 * NG))
    assert NZ // 2 + 6 <= held < NZ + 6   # the halves take one slab, the block more
    rng = np.random.default_rng(5)
    cs = (NX + 2 * NG, NY + 2 * NG, NZ + 2 * NG)
    st = {}
    for k in gpu.Solver.STATE:
        sh = tuple(n + (k == f) for n, f in zip(cs, ("bi", "bj", "bk")))
        lo, hi = (.5, 1.5) if k in ("rho", "p") else (-.5, .5)
        st[k] = np.asfortranarray(rng.uniform(lo, hi, sh[::-1]).T)
    whole = _eijk(NZ, st, recon)
    h = NZ // 2
    for z0 in (0, h):
        part = {k: np.asfortranarray(a[:, :, z0:z0 + h + 2 * NG + (k == "bk")]) for k, a in st.items()}
        e = _eijk(h, part, recon)
        for k, n in (("ei", h + 1), ("ej", h + 1), ("ek", h)):
            assert np.array_equal(e[k], whole[k][:, :, z0:z0 + n]), (k, z0)
