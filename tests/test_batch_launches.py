"""Launches of a batch whose trees differ much in length, without a device."""

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
