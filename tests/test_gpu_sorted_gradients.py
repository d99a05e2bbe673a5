"""Gradients gathered by cell (the cells' programs reach as far as the taps),
against the same points a few at a time with the whole program: bit for bit, by
both rules, for points inside, around and far outside the scene, all in one cell,
NaN and infinite, and for steps below and beyond the reach that is gathered.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PRIMS = 700          # 1399 entries: gathered from 16385 points on
N = 40_003


def _points(name):
    rng = np.random.default_rng(9)
    x = rng.uniform(-7.0, 7.0, (N, 3)).astype(np.float32)
    if name == "far":
        x[::3] *= np.float32(4.0)
        x[1::1000] *= np.float32(1e4)
        x[5], x[6], x[7] = np.nan, np.inf, (-np.inf, 0.0, 1.0)
        x[N - 1] = np.nan
    if name == "one_cell":
        x[:] = np.float32([0.3, -0.2, 0.1])
        x[:, 0] += rng.uniform(0.0, 1e-3, N).astype(np.float32)
    return x


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("central", [False, True])
@pytest.mark.parametrize("name,h", [("uniform", 1e-4), ("uniform", 0.1), ("uniform", 0.5), ("far", 1e-4), ("one_cell", 1e-3)])
def test_gathered_gradients(gpu, name, h, central, fast):
    from tangerine_amd import scenes, trace
    prog = scenes.build_sdf(scenes.random_csg_spec(12, PRIMS)).program()
    x = _points(name)
    got = trace.gradient(prog, x, h=h, central=central, fast=fast)
    ref = np.concatenate([trace.gradient(prog, x[i:i + 16_000], h=h, central=central, fast=fast) for i in range(0, N, 16_000)])
    nan = np.isnan(ref)
    assert np.array_equal(got.view(np.uint32)[~nan], ref.view(np.uint32)[~nan])
    assert np.all(np.isnan(got[nan]))
