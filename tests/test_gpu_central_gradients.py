"""Central differences: six taps to a point, three to a lane or one to a lane of a
split program.  Equal to the oracle's bits at the edges of a wave's points (10 split, 32
else) and of a workgroup's, and gathered by cell equal to the same points a few at a
time.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTS = [1, 9, 10, 11, 31, 32, 33, 127, 128, 129, 1001]


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("prims", [1, 3, 40, 300])  # one primitive: no treelets to split
def test_counts(gpu, oracle, prims):
    from tangerine_amd import scenes, trace
    node = scenes.build_sdf(scenes.random_csg_spec(70 + prims, prims))
    prog, words = node.program(), node.compile()
    x = np.random.default_rng(prims).uniform(-5.0, 5.0, (max(COUNTS), 3)).astype(np.float32)
    want = _bits(oracle.gradient_central(words, x, 1e-3))
    for n in COUNTS:
        assert np.array_equal(_bits(trace.gradient(prog, x[:n], h=1e-3, central=True)), want[:n]), n


@pytest.mark.parametrize("fast", [False, True])
def test_many(gpu, fast):
    """Past the split (16384 points) and gathered, against parts that are split."""
    from tangerine_amd import scenes, trace
    x = np.random.default_rng(3).uniform(-6.0, 6.0, (160_001, 3)).astype(np.float32)
    for prims in (3, 64, 700):
        prog = scenes.build_sdf(scenes.random_csg_spec(80 + prims, prims)).program()
        want = np.concatenate([trace.gradient(prog, x[i:i + 4000], central=True, fast=fast) for i in range(0, len(x), 4000)])
        for n in (4097, 16_385, 40_003, 160_001):
            assert np.array_equal(_bits(trace.gradient(prog, x[:n], central=True, fast=fast)), _bits(want[:n])), (prims, n)
