"""Culled exports from one program per tile against the block evaluators (a mesher
whose culled launch shape was set): the same kept bricks, the same number added by
the certificate and of tiles evaluated, the same mesh bytes; grids that end inside a
tile, a block of tiles and a workgroup of bricks.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, (1, 1, 1)), (4, (7, 9, 16)), (33, (40, 33, 65)), (256, (129, 96, 71)), (900, (64, 30, 41))]


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("surrogate", [False, True])
@pytest.mark.parametrize("prims,cells", SIZES, ids=[f"{p}-{c[0]}x{c[1]}x{c[2]}" for p, c in SIZES])
def test_culled_tiles_match_blocks(gpu, prims, cells, surrogate, fast):
    from tangerine_amd import scenes
    from tangerine_amd.export import Mesher
    from tangerine_amd.surrogate import Surrogate
    prog = scenes.build_sdf(scenes.random_csg_spec(prims, prims)).program()
    step = float(np.float32(12.0 / max(cells)))
    grid = (-6.0, -6.0, -6.0), (step,) * 3, cells
    s = None
    if surrogate:
        s = Surrogate((-6.5,) * 3, 13.0, seed=2)
        s.fit(prog, samples=16384, calib_samples=2000, epochs=1)
    out = []
    for by_blocks in (False, True):
        m = Mesher()
        if by_blocks:
            m.set_culled_tuning(4, 4, 6)
        for _ in range(2):
            st = m.export_culled(prog, s, *grid, fast=fast)
        assert (st["block_workgroups"] > 0) == by_blocks
        v, t = m.mesh()
        out.append((v.tobytes(), t.tobytes(), m.brick_flags().tobytes(), st["bricks_flagged"], st["bricks_certified"],
                    st["tiles_evaluated"], st["exact_evals"], st["cull_threshold"]))
        m.close()
    assert out[0] == out[1]
    if s is not None:
        s.close()
