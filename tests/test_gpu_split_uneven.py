"""Programs split over a workgroup whose subtrees cut unevenly: the finer upper
treelets give the oracle's values, bit for bit, where a cut operand meets an uncut
one, where a stage is wider than the workgroup, and with several stages above."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prims", [20, 49, 97, 120, 300, 1500])
def test_uneven_trees(gpu, oracle, prims):
    from tangerine_amd import scenes
    node = scenes.build_sdf(scenes.random_csg_spec(prims + 7, prims))
    prog, words = node.program(), node.compile()
    x = np.random.default_rng(prims).uniform(-7.0, 7.0, (259, 3)).astype(np.float32)
    ref = np.ascontiguousarray(oracle.interp_words(words, x), dtype=np.float32)
    for n in (1, 65, 259):
        got = np.ascontiguousarray(prog.eval_points(x[:n]), dtype=np.float32)
        assert np.array_equal(got.view(np.uint32), ref[:n].view(np.uint32)), n
