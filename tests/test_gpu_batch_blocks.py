"""Batches whose trees go through the block queue, alone and beside trees that are
evaluated from tile programs: every sample and mesh equals the tree's single export
by the other evaluator, and the count of queue items and tiles says which went where.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def _chain(levels):
    """At 15 levels to a treelet, 700 have too many stages for tile programs (more
    than 32) and go by blocks on every grid; 300 have not."""
    spec = []
    for k in range(levels):
        spec += [("sphere", 0.3 + 0.01 * (k % 50)), ("move", -4.0 + 0.2 * (k % 40), 0.1 * (k % 7), 0.01 * (k % 90))]
    return spec + [("diff",) if k % 3 else ("union",) for k in range(levels - 1)]


def _grid(cells):
    step = float(np.float32(12.0 / max(cells)))
    return (-6.0,) * 3, (step,) * 3, cells


def _tiles(cells):
    return [c // 8 + 1 for c in cells]


def _units(cells, by_blocks):
    t = _tiles(cells)
    return int(np.prod([-(-n // 4) for n in t] if by_blocks else t))


# (program, cells, by blocks): the 2048-primitive tree is past the tile programs'
# line (53^3 tiles of 4095 + 6144 entries), and prunes by treelets all the same
MIXED = [(("random", 5), (40, 33, 21), False), (("chain", 700), (50, 41, 37), True), (("random", 200), (96, 96, 96), False),
         (("random", 2048), (420, 420, 420), True), (("random", 1), (1, 1, 1), False), (("chain", 300), (9, 70, 8), False)]


def _program(kind, n):
    from tangerine_amd import scenes
    return scenes.build_sdf(_chain(n) if kind == "chain" else scenes.random_csg_spec(60 + n, n)).program()


def _single(prog, grid, by_blocks, fast):
    from tangerine_amd.export import Mesher
    m = Mesher()
    if by_blocks:
        m.set_tuning(4, 2, 8, 0)
    m.export(prog, *grid, fast=fast)
    v, t = m.mesh()
    out = _bits(m.grid()), v.tobytes(), t.tobytes()
    m.close()
    return out


def _check(b, progs, parts, fast, tag):
    for i, (_, cells, blocks) in enumerate(parts):
        m = b.mesher(i)
        want = _single(progs[i], _grid(cells), not blocks, fast)  # (a chain goes by blocks either way)
        v, t = m.mesh()
        assert np.array_equal(_bits(m.grid()), want[0]), (tag, i)
        assert v.tobytes() == want[1] and t.tobytes() == want[2], (tag, i)


@pytest.mark.parametrize("fast", [False, True])
def test_mixed_batch(gpu, fast):
    """Queue items and tile jobs side by side, in two orders in the same buffers, and
    their replays."""
    from tangerine_amd.batch import Batch
    parts = list(MIXED)
    progs = [_program(*p) for p, _, _ in parts]
    b = Batch()
    for rep in range(2):
        st = b.export(progs, [_grid(c) for _, c, _ in parts], fast=fast)
        assert st["blocks"] == sum(_units(c, k) for _, c, k in parts)
        assert st["max_len"] > 0 and st["exact_evals"] > 0
        _check(b, progs, parts, fast, rep)
        parts, progs = parts[::-1], progs[::-1]
    for _ in range(2):
        assert b.replay() > 0
    parts, progs = parts[::-1], progs[::-1]
    _check(b, progs, parts, fast, "replay")
    b.close()


@pytest.mark.parametrize("tuned", [False, True])
def test_batch_of_block_trees(gpu, tuned):
    """No tile job: the queue alone, untuned (trees that cannot go by tiles) and, for
    every tree, after a launch shape was set."""
    from tangerine_amd.batch import Batch
    parts = [p for p in MIXED if tuned or p[2]]
    parts = [(p, c, True) for p, c, _ in parts]
    progs = [_program(*p) for p, _, _ in parts]
    b = Batch()
    for shape in [(2, 2, 3), (8, 4, 2)] if tuned else [None]:
        if shape:
            b.set_tuning(*shape)
        st = b.export(progs, [_grid(c) for _, c, _ in parts])
        assert st["blocks"] == sum(_units(c, True) for _, c, _ in parts)
        _check(b, progs, parts, False, shape)
        assert b.replay() > 0
    b.close()
