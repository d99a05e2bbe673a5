"""Routes of calls whose program no cell prunes, or hardly any: they go as they would
without cells where cells only cost.  Without a device: what is launched tells."""

import pytest

from tests.fake_device import run

TREES = """
from tangerine_amd import trace
def tree(kind, n):
    "random tree; with an ellipsoid (never pruned); every operator a blend of `kind` units"
    spec = scenes.random_csg_spec(1, n)
    if kind == "ellipsoid":
        spec[next(i for i, t in enumerate(spec) if t[0] in scenes.PRIMITIVES)] = ("ellipsoid", 0.5, 0.7, 0.9)
    elif kind != "random":
        spec = [("blend_union", float(kind)) if t[0] in scenes.SET_OPS else t for t in spec]
    return scenes.build_sdf(spec).program()
"""


@pytest.mark.parametrize("kind,prims,groups", [
    ("ellipsoid", 64, (True, False)), ("ellipsoid", 256, (True, False)), ("2", 64, (True, False)), ("2", 256, (True, False)),
    ("8", 256, (True, False)), ("random", 1, (False, False)), ("random", 2, (True, False)), ("random", 3, (True, False)), ("random", 4, (True, False)), ("random", 8, (True, True)),
    ("0.1", 256, (True, True)), ("random", 16, (True, True)), ("random", 64, (True, True)),
    ("random", 256, (True, True)), ("random", 2048, (True, True))])
def test_frames(kind, prims, groups):
    """Small frames go on in groups of lanes whatever the program of 2 primitives or
    more (their waves do not fill the GPU), large ones only where cells prune; unpruned
    renders never."""
    run(TREES + f"""
p = tree({kind!r}, {prims})
tr = trace.Tracer()
for (w, h), want in zip([(320, 180), (1920, 1080)], {groups!r}):
    cam = trace.look_at((9, 6, 5), width=w, height=h)
    launches()
    tr.render(p, cam)
    assert ran("k_trace_groups", launches()) == want, (w, h)
    tr.render(p, cam, prune=False)
    assert not ran("k_trace_groups", launches())
""")


@pytest.mark.parametrize("kind,prims,points,gradients", [
    ("random", 256, {300_000: False, 600_000: True, 2_000_000: True}, {50_000: False, 200_000: True}),
    ("random", 64, {2_000_000: False}, {100_000: False, 1_000_000: True}),
    ("2", 256, {600_000: False, 2_000_000: False}, {100_000: False, 1_000_000: False}),
    ("8", 256, {600_000: False, 2_000_000: False}, {100_000: False, 1_000_000: False}),
    ("8", 1024, {150_000: False, 2_000_000: False}, {50_000: False, 1_000_000: False}),
    ("0.5", 256, {600_000: False, 2_000_000: True}, {100_000: False, 1_000_000: True})])
def test_points_and_gradients(kind, prims, points, gradients):
    run(TREES + f"""
p = tree({kind!r}, {prims})
for n, want in {points!r}.items():
    x = np.zeros((n, 3), np.float32)
    launches()
    p.eval_points(x)
    assert ran("k_eval_points_sorted", launches()) == want, n
for n, want in {gradients!r}.items():
    x = np.zeros((n, 3), np.float32)
    for central in (False, True):
        launches()
        trace.gradient(p, x, central=central)
        assert ran("k_gradient_sorted", launches()) == want, (n, central)
""")


@pytest.mark.parametrize("kind,prims,casts", [
    ("random", 256, {(64, 100): True, (50_000, 100): True, (1_000_000, 100): True, (50_000, 12): True, (50_000, 1): False,
                     (64, 1): False, (400_000, 6): False}),
    ("random", 64, {(64, 100): True, (100_000, 100): True, (50_000, 12): False, (1_000_000, 100): False}),
    ("1", 64, {(4096, 100): True, (200_000, 100): False}),
    ("8", 256, {(64, 100): False, (4096, 100): False, (50_000, 100): False}),
    ("ellipsoid", 256, {(4096, 100): False})])
def test_ray_casts(kind, prims, casts):
    run(TREES + f"""
p = tree({kind!r}, {prims})
for (n, steps), want in {casts!r}.items():
    s = np.full((n, 3), 9.0, np.float32)
    launches()
    trace.raymarch(p, s, -s, max_steps=steps)
    calls = launches()
    assert ran("k_march", calls) == want and ran("k_trace", calls) != want, (n, steps)
""")


@pytest.mark.parametrize("kind,prims,clouds", [
    ("random", 256, {(32, 0): False, (120, 0): True, (120, 2): True}), ("random", 16, {(200, 0): True, (120, 2): True}),
    ("random", 10, {(120, 0): False, (160, 6): True}), ("random", 28, {(120, 0): False, (120, 6): True}),
    ("0.5", 256, {(120, 0): True, (120, 2): False, (200, 2): True}), ("8", 64, {(120, 0): False, (120, 2): False}),
    ("8", 256, {(120, 0): False, (200, 2): False}), ("ellipsoid", 256, {(120, 0): False})])
def test_point_clouds(kind, prims, clouds):
    run(TREES + f"""
from tangerine_amd.export import Mesher
p = tree({kind!r}, {prims})
m = Mesher()
for (n, steps), want in {clouds!r}.items():
    launches()
    m.export_points(p, (-6.0,) * 3, (6.0,) * 3, (float(np.float32(12.0 / n)),) * 3, refine_iterations=steps)
    calls = launches()
    assert ran("k_cloud_select_tiles", calls) == want and ran("k_prune", calls) == want, (n, steps)
""")


@pytest.mark.parametrize("kind,tiles", [("random", True), ("2", True), ("8", False)])
def test_culled_exports(kind, tiles):
    run(TREES + f"""
from tangerine_amd.export import Mesher
m = Mesher()
m.export_culled(tree({kind!r}, 256), None, *scenes.grid_for(-6.0, 6.0, 128))
assert ran("k_certify_tiles", launches()) == {tiles}
""")
