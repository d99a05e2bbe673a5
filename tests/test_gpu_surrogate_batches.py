"""A fit of several batches and epochs against the same steps taken on the host: every
batch's samples are those of the training order, and every step is numbered through.

As in the test of one batch the field has no surface in the domain.  A batch's mean
loss differs from another's by about a hundredth (16384 samples), a hundred times what
a step's loss may be off.
"""

import numpy as np
import pytest

from tests.test_gpu_surrogate_fit import LO, SEED, SIZE, _uniform01

pytestmark = pytest.mark.gpu

BATCH = 16384


@pytest.mark.parametrize("batches,epochs", [(2, 3), (3, 2), (5, 1)])
def test_fit_of_batches_matches_host_steps(gpu, oracle, batches, epochs):
    from tangerine_amd import sdf
    from tangerine_amd.surrogate import Surrogate
    program = sdf.sphere(8.0).move(1.0, 0.5, 0.25).program()
    n = batches * BATCH
    s = Surrogate(LO, SIZE, sigma=1.0, clamp=4.0, seed=SEED)
    p, _ = s.params()
    i = np.arange(n, dtype=np.uint64)[:, None] * np.uint64(8) + np.arange(3, dtype=np.uint64)
    x = (np.float32(LO[0]) + np.float32(SIZE) * _uniform01(i)).astype(np.float32)
    target = program.eval_points(x)
    order = oracle.training_order(SEED, n)
    assert np.array_equal(np.sort(order), np.arange(n))

    st = s.fit(program, samples=n, calib_samples=64, epochs=epochs)
    assert st["steps"] == epochs * batches and st["surface_vertices"] == 0
    got, _ = s.params()
    losses = s.loss_log()
    assert len(losses) == epochs * batches

    ref = p.astype(np.float64)
    m, v = np.zeros_like(ref), np.zeros_like(ref)
    for k in range(1, epochs * batches + 1):
        at = order[(k - 1) % batches * BATCH:][:BATCH]
        s.set_params(ref.astype(np.float32))
        loss, g = s.gradients(x[at], target[at])
        assert losses[k - 1] == pytest.approx(loss, rel=1e-4), k
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * np.square(g, dtype=np.float64)
        lr = 2e-3 * (0.05 + 0.475 * (1.0 + np.cos(np.pi * k / (epochs * batches))))
        ref -= lr * (m / (1.0 - 0.9 ** k)) / (np.sqrt(v / (1.0 - 0.999 ** k)) + 1e-8)
    move = ref - p
    assert np.linalg.norm(got - p - move) <= 2e-2 * np.linalg.norm(move)
    s.close()
