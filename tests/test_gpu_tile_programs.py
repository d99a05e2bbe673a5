"""Exports evaluated from one program per 8^3-sample tile (grids whose tiles x
program entries are few) against the block evaluators and the oracle.

A mesher whose launch shape was set evaluates by blocks; a fresh one takes
tile programs where they fit.  Both run value-exact pruned programs, so the
samples and the mesh are the same bits.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def _export(prog, grid, by_blocks, fast=False):
    from tangerine_amd.export import Mesher
    m = Mesher()
    if by_blocks:
        m.set_tuning(4, 2, 0, 8)
    st = m.export(prog, *grid, fast=fast)
    v, t = m.mesh()
    out = _bits(m.grid()), v.tobytes(), t.tobytes(), st
    m.close()
    return out


def _grid(lo, hi, cells):
    step = float(np.float32((hi - lo) / max(cells)))
    return (float(np.float32(lo)),) * 3, (step,) * 3, cells


# edges of a tile (8 samples = 7 cells), of a workgroup's tiles and cells, one
# entry, and the programs' edges: 64-entry chunks, overflowing pool guesses
SIZES = [(1, (1, 1, 1)), (1, (7, 8, 9)), (2, (8, 1, 15)), (3, (33, 40, 17)), (32, (64, 64, 64)), (33, (71, 50, 23)),
         (256, (96, 97, 95)), (700, (40, 33, 60)), (2048, (64, 64, 64))]


@pytest.mark.parametrize("prims,cells", SIZES, ids=[f"{p}-{c[0]}x{c[1]}x{c[2]}" for p, c in SIZES])
@pytest.mark.parametrize("fast", [False, True])
def test_tile_programs_match_blocks(gpu, prims, cells, fast):
    from tangerine_amd import scenes
    prog = scenes.build_sdf(scenes.random_csg_spec(prims + 1, prims)).program()
    g = _grid(-6.0, 6.0, cells)
    a, b = _export(prog, g, False, fast), _export(prog, g, True, fast)
    assert a[3]["block_workgroups"] == 0 and b[3]["block_workgroups"] > 0  # the two paths ran
    assert np.array_equal(a[0], b[0])
    assert a[1] == b[1] and a[2] == b[2]
    assert a[3]["exact_evals"] == 512 * int(np.prod([c // 8 + 1 for c in cells]))
    if prims > 30:
        assert a[3]["flops"] <= b[3]["flops"] * 1.05  # pruned as far as the block evaluators prune


def _operator_specs():
    specs = []
    for op in ("union", "inter", "diff", "blend_union", "blend_inter", "blend_diff"):
        tok = (op, 0.2) if op.startswith("blend") else (op,)
        specs.append([("sphere", 1.0), ("move", -3.0, 0.0, 0.0), ("box", 0.5, 0.7, 0.9), ("move", 3.0, 0.5, 0.0),
                      tok, ("torus", 1.0, 0.3), ("move", 0.0, -3.0, 1.0), tok])
    # right-leaning: operands swapped, several stages of treelets; 700 levels
    # exceed the stages and are pruned by one wave per block group
    for n in (40, 70, 700):
        chain = []
        for k in range(n):
            chain += [("sphere", 0.3 + 0.01 * (k % 50)), ("move", -4.0 + 0.2 * (k % 40), 0.1 * (k % 7), 0.01 * (k % 90))]
        specs.append(chain + [("diff",) if k % 3 else ("blend_union", 0.1) if n < 100 else ("union",) for k in range(n - 1)])
    specs.append([("box", 1.0, 0.5, 0.7), ("flate", 0.2), ("sphere", 0.8), ("scale", 1.5), ("move", 1.0, 0.0, 0.0),
                  ("blend_diff", 0.25), ("flate", 0.05)])
    return specs


@pytest.mark.parametrize("k", range(10))
def test_tile_programs_on_operator_cases(gpu, oracle, k):
    """Dropped and kept operands, negation, the +0.0 flag, swapped operands,
    unary operators: blocks and the oracle's interpreter give the same bits."""
    from tangerine_amd import scenes
    spec = _operator_specs()[k]
    node = scenes.build_sdf(spec)
    g = _grid(-5.0, 5.0, (50, 41, 37))
    a, b = _export(node.program(), g, False), _export(node.program(), g, True)
    assert np.array_equal(a[0], b[0]) and a[1:3] == b[1:3]
    expect, _ = oracle.grid_interp(node.compile(), *g, threads=8)
    assert np.array_equal(a[0], _bits(expect.ravel()))


def test_batch_of_tile_and_block_trees(gpu):
    """A batch with trees of both kinds (a fine grid of a long program is
    evaluated by blocks) equals every tree's single export, replays included."""
    from tangerine_amd import scenes
    from tangerine_amd.batch import Batch
    parts = [(5, (40, 33, 21)), (1, (1, 1, 1)), (2048, (300, 300, 290)), (200, (96, 96, 96)), (17, (9, 70, 8))]
    progs = [scenes.build_sdf(scenes.random_csg_spec(50 + i, n)).program() for i, (n, _) in enumerate(parts)]
    grids = [_grid(-6.0, 6.0, c) for _, c in parts]
    b = Batch()
    for rep in range(2):  # the second export in the first one's buffers
        st = b.export(progs, grids)
        for i, g in enumerate(grids):
            m = b.mesher(i)
            want = _export(progs[i], g, True)
            v, t = m.mesh()
            assert np.array_equal(_bits(m.grid()), want[0]), (rep, i)
            assert v.tobytes() == want[1] and t.tobytes() == want[2], (rep, i)
            assert m.stats()["exact_evals"] > 0
        progs, grids = progs[::-1], grids[::-1]
    for _ in range(2):
        assert b.replay() > 0
    assert np.array_equal(_bits(b.mesher(0).grid()), _export(progs[::-1][0], grids[::-1][0], True)[0])
    b.close()
