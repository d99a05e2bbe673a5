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
