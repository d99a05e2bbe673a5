"""Point clouds through one program per 8^3 cells against the whole program at
every cell (TG_FLAG_NO_PRUNE): the same points, bit for bit, on grids that end
inside a tile, with steps of their own per axis, with and without refinement.
"""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cloud(m, prog, lo, hi, step, iterations, flags):
    from tangerine_amd import _lib
    f3 = lambda v: (C.c_float * 3)(*v)
    _lib.check(m.lib.tg_mesher_export_points(m.h, prog.handle, f3(lo), f3(hi), f3(step), iterations, flags), "points")
    return m.mesh()[0].view(np.uint32)


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("prims,cells,iterations", [
    (256, (65, 63, 65), 0), (256, (64, 33, 72), 2), (256, (9, 400, 23), 4), (512, (47, 48, 49), 1), (97, (121, 60, 57), 3)])
def test_tile_programs_keep_the_points(gpu, prims, cells, iterations, fast):
    from tangerine_amd import _lib, scenes
    from tangerine_amd.export import Mesher
    prog = scenes.build_sdf(scenes.random_csg_spec(prims + 3, prims)).program()
    assert int(np.prod(cells)) * (2 * prims - 1) * (1 + iterations) >= 120 << 20   # past the rule's line
    lo, hi = (-5.5, -6.0, -5.0), (6.0, 5.0, 5.75)
    step = [float(np.float32((h - l) / (n - 0.5))) for l, h, n in zip(lo, hi, cells)]
    flags = _lib.TG_FLAG_FAST if fast else 0
    m = Mesher()
    ref = _cloud(m, prog, lo, hi, step, iterations, flags | _lib.TG_FLAG_NO_PRUNE)
    got = _cloud(m, prog, lo, hi, step, iterations, flags)
    assert len(ref) > 500 and np.array_equal(got, ref)
    m.close()
