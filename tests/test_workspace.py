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


@pytest.mark.parametrize("device_pointers", [False, True])
def test_point_queries_without_room_for_cells(device_pointers):
    """Queries that would be gathered by cell but find no memory for that run the whole
    program, which needs none beside the points and results of a host call."""
    run(f"""
p = program(256)
n = 700_000
x, out = np.zeros((n, 3), np.float32), np.zeros(n, np.float32)
def query():
    if {device_pointers}:
        _lib.check(lib.tg_eval_points_device(p.handle, x.ctypes.data, n, out.ctypes.data, 0, None), "query")
    else:
        p.eval_points(x)
room = 0 if {device_pointers} else 16 * n + 4096
fake.fake_limit(fake.fake_used() + room)
launches()
query()
calls = launches()
assert ran("k_eval_points", calls) and not ran("sorted", calls) and not ran("k_prune", calls)
fake.fake_limit(1 << 38)
query()
assert ran("k_eval_points_sorted", launches())
""")


def test_gradients_without_room_for_cells():
    run("""
from tangerine_amd import trace
p = program(256)
n = 300_000
x = np.zeros((n, 3), np.float32)
fake.fake_limit(fake.fake_used() + 24 * n + 4096)
launches()
trace.gradient(p, x)
calls = launches()
assert ran("k_gradient", calls) and not ran("sorted", calls)
""")


def test_idle_workspaces_are_given_back():
    """What queries left allocated goes where an allocation would fail without it."""
    run("""
from tangerine_amd.export import Mesher
base = fake.fake_used()
p = program(256)
p.eval_points(np.zeros((700_000, 3), np.float32))
kept = fake.fake_used() - base
assert kept > (1 << 20)
fake.fake_peak()
m = Mesher()
m.export(p, *scenes.grid_for(-6.0, 6.0, 100))
need = fake.fake_peak() - base - kept
m.close()
fake.fake_limit(base + need + kept // 2)
m = Mesher()
m.export(p, *scenes.grid_for(-6.0, 6.0, 100))
""")
