"""Training steps (two groups of points to a workgroup, block sums, Adam) against
the same steps taken on the host with the gradients of single groups.

The field has no surface in the domain, so that every sample is uniform and its
hash can be repeated here.  Per step the mean loss agrees to 1e-4 (sums of 16384
float squares in another order), and after three steps the movement of all
parameters to 2e-2 of its norm: the bar of the gradients themselves, which Adam
divides by their own size.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LO, SIZE, SEED, N = (-1.0, -1.0, -1.0), 2.0, 21, 16384


def _uniform01(i):
    with np.errstate(over="ignore"):
        x = np.uint64(SEED) * np.uint64(0x9E3779B97F4A7C15) + i.astype(np.uint64)
        x ^= x >> np.uint64(33)
        x *= np.uint64(0xFF51AFD7ED558CCD)
        x ^= x >> np.uint64(33)
        x *= np.uint64(0xC4CEB9FE1A85EC53)
        x ^= x >> np.uint64(33)
    u = (x & np.uint64(0xFFFFFFFF)) >> np.uint64(8)
    return (u.astype(np.float32) + np.float32(0.5)) * np.float32(1.0 / 16777216.0)


def test_fit_steps_match_host_steps(gpu):
    from tangerine_amd import sdf
    from tangerine_amd.surrogate import Surrogate
    program = sdf.sphere(8.0).move(1.0, 0.5, 0.25).program()
    s = Surrogate(LO, SIZE, sigma=1.0, clamp=4.0, seed=SEED)
    p, _ = s.params()
    i = np.arange(N, dtype=np.uint64)[:, None] * np.uint64(8) + np.arange(3, dtype=np.uint64)
    x = (np.float32(LO[0]) + np.float32(SIZE) * _uniform01(i)).astype(np.float32)
    target = program.eval_points(x)
    assert np.ptp(target) > 1.0 and np.all(target < 0.0)

    epochs, batches = 3, 1
    st = s.fit(program, samples=N, calib_samples=64, epochs=epochs)
    assert st["steps"] == epochs and st["surface_vertices"] == 0
    got, _ = s.params()
    losses = s.loss_log()

    ref = p.astype(np.float64)
    m, v = np.zeros_like(ref), np.zeros_like(ref)
    for k in range(1, epochs * batches + 1):
        s.set_params(ref.astype(np.float32))
        loss, g = s.gradients(x, target)
        assert losses[k - 1] == pytest.approx(loss, rel=1e-4), k
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * np.square(g, dtype=np.float64)
        lr = 2e-3 * (0.05 + 0.475 * (1.0 + np.cos(np.pi * k / epochs)))
        ref -= lr * (m / (1.0 - 0.9 ** k)) / (np.sqrt(v / (1.0 - 0.999 ** k)) + 1e-8)
    move = ref - p
    assert np.linalg.norm(got - p - move) <= 2e-2 * np.linalg.norm(move)
    s.close()
