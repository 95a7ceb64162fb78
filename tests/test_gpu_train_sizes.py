"""The training kernel's chunks: a batch is cut into 64 runs of consecutive
samples, 16 at a time.  Sizes where a run is empty, partly filled, or needs
several tiles, against a binary64 gradient (torch autograd on the CPU).

The kernel adds fp32 products: a unit's sum of at most 41, three layers deep,
then at most n/64 + 64 samples' terms in sequence -- about 150 + n/64 roundings
of 6e-8 each, so 2e-5 of the gradient's norm bounds the difference with a
factor of two to spare at the largest n.
"""
import numpy as np
import pytest
import torch

from mhd3d_mpi_fortran_amd import gpu, ics
from mhd3d_mpi_fortran_amd import surrogate as sg

pytestmark = pytest.mark.gpu


def _reference(w, s):
    p = torch.tensor(w.astype(np.float64), requires_grad=True)
    x, t = (torch.tensor(a.astype(np.float64)) for a in (s[:, :40], s[:, 40:]))
    x5 = x.reshape(-1, 8, 5)
    lin = (-x5[:, :, 0] + 7. * x5[:, :, 1] + 7. * x5[:, :, 2] - x5[:, :, 3]) / 12.
    gate = (x5[:, :, :-2] - 2. * x5[:, :, 1:-1] + x5[:, :, 2:]).abs().amax(dim=2)
    h, o = x, 0
    for rows, cols in ((32, 40), (32, 32), (16, 32)):
        h = h @ p[o:o + rows * cols].reshape(rows, cols).T + p[o + rows * cols:o + rows * cols + rows]
        o += rows * cols + rows
        if rows == 32:
            h = h * torch.sigmoid(1.702 * h)
    loss = ((lin.repeat(1, 2) + gate.repeat(1, 2) * h - t) ** 2).mean()
    loss.backward()
    return float(loss.detach()), p.grad.numpy()


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 1000, 1024, 1025, 2500])
def test_gradient_at_chunk_edges(n):
    rng = np.random.default_rng(n)
    w = rng.uniform(-.3, .3, sg.NPARAM).astype(np.float32)
    s = rng.uniform(-1., 1., (n, sg.NSAMPLE)).astype(np.float32)
    solver = gpu.Solver(gpu.make_params(8, 8, 8), ics.Grid(8, 8, 8))
    loss, g = sg.grad(solver, w, s)
    solver.close()
    ref_loss, ref = _reference(w, s)
    assert abs(loss - ref_loss) <= 2e-5 * ref_loss
    assert np.linalg.norm(g - ref) <= 2e-5 * np.linalg.norm(ref)
