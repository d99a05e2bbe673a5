"""Calls whose usual route needs more memory than there is take the one that needs
little, without a device: each runs within what it needed by that route."""

import pytest

from tests.fake_device import run


@pytest.mark.parametrize("culled", [False, True])
@pytest.mark.parametrize("headroom", [0, 1 << 20, 1 << 22, 1 << 24])
def test_exports_go_by_blocks(culled, headroom):
    """Within the memory of an export by blocks, and a little more: the passes over
    tiles find no room at their start, or the later stages none behind them."""
    run(f"""
from tangerine_amd.export import Mesher
p = program(1500)
g = scenes.grid_for(-6.0, 6.0, 200)
def export(blocks):
    m = Mesher()
    if blocks:
        m.set_tuning(4, 2, 8, 8)
        m.set_culled_tuning(4, 4, 6)
    fake.fake_peak()
    launches()
    st = m.export_culled(p, None, *g) if {culled} else m.export(p, *g)
    return m, launches()
base = fake.fake_used()
m, calls = export(True)
need = fake.fake_peak() - base
m.close()
m, calls = export(False)
assert ran("k_eval_tile_programs", calls)
more = fake.fake_peak() - base
m.close()
assert more > need + (1 << 24), (need, more)
fake.fake_limit(base + need + {headroom})
m, calls = export(False)
assert not ran("k_eval_tile_programs", calls)
fake.fake_limit(1 << 38)
m.export(p, *g)
assert ran("k_eval_tile_programs", launches())
""")


def test_point_clouds_take_the_whole_program():
    run("""
from tangerine_amd.export import Mesher
p = program(256)
def cloud(m):
    fake.fake_peak()
    launches()
    m.export_points(p, (-6.0,) * 3, (6.0,) * 3, (0.1,) * 3, refine_iterations=2)
    return launches()
base = fake.fake_used()
m = Mesher()
assert ran("k_cloud_select_tiles", cloud(m))
m.close()
base = fake.fake_used()
fake.fake_limit(base + 121 ** 3 * 8 + (1 << 20))  # flags and ranks
m = Mesher()
calls = cloud(m)
assert ran("k_cloud_select", calls) and not ran("tiles", calls)
""")


@pytest.mark.parametrize("headroom", [0, 1 << 18, 1 << 23])
def test_ray_casts_take_the_whole_program(headroom):
    run(f"""
from tangerine_amd import trace
p = program(256)
s = np.full((5000, 3), 9.0, np.float32)
fake.fake_limit(fake.fake_used() + 5000 * 41 + 512 + {headroom})
launches()
trace.raymarch(p, s, -s)
calls = launches()
assert ran("k_trace", calls) and not ran("k_march", calls)
assert fake.fake_pending() == 0
fake.fake_limit(1 << 38)
trace.raymarch(p, s, -s)
assert ran("k_march", launches())
""")


BATCH = """
from tangerine_amd.batch import Batch
def batch(trees, cells, p, blocks):
    b = Batch()
    if blocks:
        b.set_tuning(4, 4, 4)  # (the shape of an untuned batch)
    fake.fake_peak()
    launches()
    st = b.export([p] * trees, [scenes.grid_for(-6.0, 6.0, cells)] * trees)
    return b, st, launches()
def units(cells):
    t = cells // 8 + 1
    return t ** 3, (-(-t // 4)) ** 3
"""


@pytest.mark.parametrize("headroom", [0, 1 << 20, 1 << 24, 1 << 27])
def test_batches_go_by_blocks(headroom):
    run(BATCH + f"""
tiles, blocks = units(150)
p = program(1500)
base = fake.fake_used()
b, st, calls = batch(32, 150, p, True)
need = fake.fake_peak() - base
assert st["blocks"] == 32 * blocks
b.close()
b, st, calls = batch(32, 150, p, False)
assert st["blocks"] == 32 * tiles and fake.fake_peak() - base > need + (1 << 27)
b.close()
fake.fake_limit(base + need + {headroom})
b, st, calls = batch(32, 150, p, False)
assert st["blocks"] == 32 * blocks and not ran("k_eval_tile_programs", calls)
assert b.replay() > 0
""")


def test_tile_programs_of_a_large_batch_are_bounded():
    """200 trees whose tile programs would take 21 GB: as many as 16 GiB hold go by
    tiles, the others by blocks."""
    run(BATCH + """
tiles, blocks = units(330)
p = program(2048)
base = fake.fake_used()
b, st, calls = batch(200, 330, p, True)
need = fake.fake_peak() - base
b.close()
b, st, calls = batch(200, 330, p, False)
by_tiles = (st["blocks"] - 200 * blocks) / (tiles - blocks)
assert by_tiles == int(by_tiles) and 0 < by_tiles < 200, by_tiles
assert fake.fake_peak() - base <= need + (17 << 30), (fake.fake_peak(), need)
assert ran("k_eval_tile_programs_multi", calls) and ran("k_eval_batch", calls)
""")


def test_what_tiles_keep_counts_towards_the_bound():
    """Tiles of wide blends keep the whole program: 250 such trees would take 40 GB."""
    run(BATCH + """
spec = [("blend_union", 8.0) if t[0] in scenes.SET_OPS else t for t in scenes.random_csg_spec(1, 600)]
p = scenes.build_sdf(spec).program()
tiles, blocks = units(250)
b, st, calls = batch(250, 250, p, False)
by_tiles = (st["blocks"] - 250 * blocks) / (tiles - blocks)
assert 0 < by_tiles < 140, by_tiles
""")
