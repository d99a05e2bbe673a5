"""Surface nets at the edges of the scanning stages' workgroups (4096 words of 64
cubes, 1024 active cubes), alone and as a batch: vertices and triangles equal to
the oracle's over the same samples, made the waiting way first and then in the room.
"""

import numpy as np
import pytest

from conftest import canonical_faces

pytestmark = pytest.mark.gpu

# cells per axis: words = sy sz ceil(sx / 64) below, at and past 4096 and 8192; one cube; thin grids
SIZES = [(64, 64, 64), (64, 64, 63), (63, 65, 64), (65, 64, 64), (130, 64, 43), (1, 1, 1), (200, 3, 2), (2, 90, 91),
         (40, 128, 32)]


def _grid(lo, hi, cells):
    step = tuple(float(np.float32((h - l) / n)) for l, h, n in zip(lo, hi, cells))
    return tuple(lo), step, tuple(cells)


def _check(oracle, mesher, grid, got):
    v, t = got
    ref_v, ref_t = oracle.surface_nets(mesher.grid(), *grid)
    assert np.array_equal(np.ascontiguousarray(v).view(np.uint32), np.ascontiguousarray(ref_v).view(np.uint32))
    assert np.array_equal(canonical_faces(t), canonical_faces(ref_t))


@pytest.mark.parametrize("cells", SIZES, ids=["x".join(map(str, c)) for c in SIZES])
def test_scan_edges(gpu, oracle, cells):
    from tangerine_amd import scenes
    from tangerine_amd.export import Mesher
    prog = scenes.build_sdf(scenes.random_csg_spec(7, 24)).program()
    grid = _grid((-4.0, -4.5, -3.5), (4.0, 3.5, 4.5), cells)
    m = Mesher()
    for _ in range(2):
        m.export(prog, *grid)
        _check(oracle, m, grid, m.mesh())
    m.close()


def test_batch_of_edges(gpu, oracle):
    from tangerine_amd import scenes
    from tangerine_amd.batch import Batch
    progs = [scenes.build_sdf(scenes.random_csg_spec(k + 1, 5 + 3 * k)).program() for k in range(len(SIZES))]
    grids = [_grid((-4.0, -4.5, -3.5), (4.0, 3.5, 4.5), c) for c in SIZES]
    b = Batch()
    for _ in range(3):
        b.export(progs, grids)
        for i, g in enumerate(grids):
            _check(oracle, b.mesher(i), g, b.mesher(i).mesh())
    # every tree's cells changed hands: rooms of other meshes
    for _ in range(2):
        b.export(progs[::-1], grids[::-1])
        for i, g in enumerate(grids[::-1]):
            _check(oracle, b.mesher(i), g, b.mesher(i).mesh())
    b.close()
