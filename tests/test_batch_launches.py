"""Launches of batches whose trees differ much in length or in route, without a device."""

import pytest

from tests.fake_device import run


@pytest.mark.parametrize("prims", [5000, 27500, 32700])
def test_column_emission_of_a_long_and_a_short_program(prims):
    """A long program emits with few waves and a large table, a short one with many
    and a small one: the shared launch holds either (at most 4 waves of 12 KiB), not
    the product of the two maxima."""
    run(f"""
from tangerine_amd.batch import Batch
def balanced(n):
    leaves = [[("sphere", 0.5), ("move", 0.01 * (k % 500), 0.1 * (k % 7), 0.0)] for k in range(n)]
    while len(leaves) > 1:
        leaves = [leaves[i] + leaves[i + 1] + [("union",)] if i + 1 < len(leaves) else leaves[i]
                  for i in range(0, len(leaves), 2)]
    return scenes.build_sdf(leaves[0]).program()
progs = [balanced({prims}), program(20)]
grids = [scenes.grid_for(-6.0, 6.0, 256), scenes.grid_for(-6.0, 6.0, 32)]
b = Batch()
b.export(progs, grids)
calls = [c for c in launches() if "k_prune_columns_multi" in c[0]]
assert calls, "no column emission"
assert max(c[3] for c in calls) <= 4 * 12288, calls
""")


def test_tuning_without_a_queue_keeps_the_shape():
    """All trees by tile programs: the queue is empty, and the launch shape that later
    batches with block trees take is not picked by the noise of its launches."""
    run("""
from tangerine_amd.batch import Batch
chain = []
for k in range(700):
    chain += [("sphere", 0.3 + 0.01 * (k % 50)), ("move", -4.0 + 0.2 * (k % 40), 0.1 * (k % 7), 0.01 * (k % 90))]
chain = scenes.build_sdf(chain + [("union",)] * 699).program()  # too many stages for tile programs
grid = scenes.grid_for(-6.0, 6.0, 50)
b = Batch()
b.export([chain], [grid])
shape = [c for c in launches() if "k_eval_batch" in c[0]]
b.export([program(30)], [grid])
launches()
r = b.autotune()
assert len(r["candidates"]) == 18 and (r["points_per_lane"], r["waves"], r["workgroups_per_cu"]) == (4, 4, 4), r
launches()
b.export([chain], [grid])
assert [c for c in launches() if "k_eval_batch" in c[0]] == shape
b.autotune()
b.close()
""")
