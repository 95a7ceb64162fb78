"""Training minibatch by minibatch against a binary64 restatement on the CPU: the
order of the samples, the gradient's mean over the batch, Adam's moments with their
corrections, the cosine schedule and the returned loss.

Tolerances.  A gradient has an error of up to 2e-5 of its norm (test_gpu_train_sizes),
about 2e-5 of their mean size an entry.  Adam divides an entry by its own size, so the
step of an entry of x mean sizes is wrong by up to 2e-5 / x of a step (at most two
steps): in the mean of squares over entries that lie evenly around zero about
4 * 2e-5, 1e-2 of the step.  So the weights' change agrees to 1e-2 of its norm.
The loss agrees to 1e-2 then as well, while a chunk of the batch left out of it or
counted twice is 1/64.
"""
import math

import numpy as np
import pytest

from mhd3d_mpi_fortran_amd import gpu, ics
from mhd3d_mpi_fortran_amd import surrogate as sg
from test_gpu_train_sizes import _reference

pytestmark = pytest.mark.gpu

N, LR = 2301, 1e-3


def restated(w, samples, epochs, batch, seed):
    n, m64 = len(samples), 2**64 - 1
    w, m, v = w.astype(np.float64), np.zeros(w.size), np.zeros(w.size)
    z, t, nb = 0xD1B54A32D192ED03 ^ seed, 0, n // batch
    for e in range(epochs):
        z = (z * 6364136223846793005 + 1442695040888963407) & m64
        mult = ((z >> 17) % n) | 1
        while math.gcd(mult, n) != 1:
            mult += 2
        first, loss = (z >> 7) % n, 0.
        for b in range(nb):
            at = (first + (b * batch + np.arange(batch)) * (mult % n)) % n
            part, g = _reference(w, samples[at])
            loss += part / nb
            t += 1
            m, v = .9 * m + .1 * g, .999 * v + .001 * g * g
            lr = LR * .5 * (1. + math.cos(math.pi * (e + b / nb) / epochs))
            w = w - lr * (m / (1. - .9**t)) / (np.sqrt(v / (1. - .999**t)) + 1e-8)
    return loss, w


# runs of 1 to 2 samples a chunk, of 4, of just one 16-sample tile, of more than one
@pytest.mark.parametrize("epochs,batch", [(1, 65), (1, 100), (2, 250), (2, 1024), (3, 1100)])
def test_training_steps(epochs, batch):
    rng = np.random.default_rng(batch)
    w0 = rng.uniform(-.3, .3, sg.NPARAM).astype(np.float32)
    samples = rng.uniform(-1., 1., (N, sg.NSAMPLE)).astype(np.float32)
    s = gpu.Solver(gpu.make_params(8, 8, 8), ics.Grid(8, 8, 8))
    sg.set_weights(s, w0)
    sg.load_samples(s, samples)
    loss = sg.train(s, epochs=epochs, batch=batch, lr=LR, seed=7)
    w = sg.get_weights(s).astype(np.float64)
    s.close()
    ref_loss, ref = restated(w0, samples, epochs, batch, 7)
    assert np.linalg.norm(w - ref) <= 1e-2 * np.linalg.norm(ref - w0)
    assert abs(loss - ref_loss) <= 1e-2 * ref_loss
