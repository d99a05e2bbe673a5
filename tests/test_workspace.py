"""Workspaces of host queries, without a device: what calls allocate, keep and give
back."""

import pytest

from tests.fake_device import run

RAYS = """
from tangerine_amd import trace
def rays(n):
    s = np.zeros((n, 3), np.float32); s[:, 0] = 9.0
    d = np.zeros((n, 3), np.float32); d[:, 0] = -1.0
    return s, d
"""


@pytest.mark.parametrize("prims", [64, 256, 300, 512])
def test_ray_casts_allocate_once(prims):
    """Later casts find the first one's buffers."""
    run(RAYS + f"""
p = program({prims})
s, d = rays(5000)
trace.raymarch(p, s, d)
assert ran("k_march", launches())
before, used = fake.fake_mallocs(), fake.fake_used()
trace.raymarch(p, s, d)
assert fake.fake_mallocs() == before and fake.fake_used() == used, (fake.fake_mallocs() - before, used)
""")


@pytest.mark.parametrize("kernel", ["k_prune_treelets", "k_prune_counts", "k_marchEN", "k_march_far"])
def test_a_failed_ray_cast_leaves_nothing_running(kernel):
    """A cast that fails behind its uploads waits for them before its buffers and the
    caller's arrays are anybody else's."""
    run(RAYS + f"""
p = program(256)
s, d = rays(5000)
trace.raymarch(p, s, d)
assert fake.fake_pending() == 0
fake.fake_fail(b"{kernel}")
try:
    trace.raymarch(p, s, d)
    raise SystemExit("no error")
except _lib.TangerineError:
    pass
assert fake.fake_pending() == 0, fake.fake_pending()
fake.fake_fail(b"")
trace.raymarch(p, s, d)
assert fake.fake_pending() == 0
""")


@pytest.mark.parametrize("kernel", ["k_eval_points_sorted", "k_point_ranks", "k_prune_treelets", "k_eval_points_split"])
def test_failed_point_queries_leave_nothing_running(kernel):
    run(f"""
p = program(256)
for n in (1000, 700_000):
    x = np.zeros((n, 3), np.float32)
    fake.fake_fail(b"{kernel}")
    launches()
    try:
        p.eval_points(x)
    except _lib.TangerineError:
        pass
    assert fake.fake_pending() == 0, (n, fake.fake_pending())
    fake.fake_fail(b"")
    p.eval_points(x)
    assert fake.fake_pending() == 0
""")
