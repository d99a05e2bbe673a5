"""tg_raymarch through cell programs (a program per lane, then the rays that
left every cell with the whole program split over a workgroup) against
tg_raymarch_static, which marches the whole program a wave: hit flags, travel
and positions are the same bits.
"""

import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rays(seed, n, spread=12.0):
    rng = np.random.default_rng(seed)
    s = rng.uniform(-spread, spread, (n, 3)).astype(np.float32)
    d = (rng.uniform(-4.0, 4.0, (n, 3)) - s).astype(np.float32)
    d[::7] = -d[::7]  # some leave the scene at once
    return s, d


def _march(fn, prog, s, d, steps, eps, far, flags):
    from tangerine_amd import _lib
    lib = _lib.load()
    n = len(s)
    hit = np.full(n, 7, dtype=np.uint8)
    t = np.full(n, np.nan, dtype=np.float32)
    pos = np.full((n, 3), np.nan, dtype=np.float32)
    fp = C.POINTER(C.c_float)
    rc = getattr(lib, fn)(prog.handle, s.ctypes.data_as(fp), d.ctypes.data_as(fp), n, steps, C.c_float(eps),
                          C.c_float(far), flags, hit.ctypes.data_as(C.POINTER(C.c_uint8)), t.ctypes.data_as(fp),
                          pos.ctypes.data_as(fp))
    assert rc == 0, lib.tg_last_error()
    return hit, t.view(np.uint32), pos.view(np.uint32)


def _same(prog, s, d, steps=100, eps=1e-3, far=math.inf, flags=0):
    a = _march("tg_raymarch", prog, s, d, steps, eps, far, flags)
    b = _march("tg_raymarch_static", prog, s, d, steps, eps, far, flags)
    assert np.array_equal(a[0], b[0])
    for x, y in zip(a[1:], b[1:]):
        # (a NaN position may carry any sign and payload)
        nan = np.isnan(y.view(np.float32))
        assert np.array_equal(nan, np.isnan(x.view(np.float32))) and np.array_equal(x[~nan], y[~nan])
    return b


# programs around the rule's smallest (112 entries), of one, two and three
# stages of treelets; counts around a wave, a workgroup of far rays, and the
# finer cells' threshold
@pytest.mark.parametrize("prims", [13, 56, 57, 80, 256, 700])
@pytest.mark.parametrize("count", [1, 63, 65, 1000, 4097])
def test_counts_and_programs(gpu, prims, count):
    from tangerine_amd import scenes
    prog = scenes.build_sdf(scenes.random_csg_spec(prims, prims)).program()
    s, d = _rays(count, count)
    hit = _same(prog, s, d)[0]
    if count > 60:
        assert 0 < hit.sum() < count


@pytest.mark.parametrize("fast", [0, 1])
@pytest.mark.parametrize("steps,eps,far", [(1, 1e-3, math.inf), (2, 1e-3, 40.0), (100, 1e-4, 40.0), (256, 0.05, 3.0),
                                           (0, 1e-3, math.inf), (100, -1.0, 20.0)])
def test_limits(gpu, fast, steps, eps, far):
    from tangerine_amd import scenes
    prog = scenes.build_sdf(scenes.random_csg_spec(3, 120)).program()
    s, d = _rays(5, 3000)
    _same(prog, s, d, steps, eps, far, fast)


def test_unusual_rays_and_programs(gpu):
    """Starts far out, at infinity, NaN, exactly on cell faces; zero and NaN
    directions; deep, swapped, unary, unprunable and unbounded programs."""
    from tangerine_amd import scenes
    s, d = _rays(9, 2000)
    s[0] = np.nan
    s[1] = np.inf
    s[2] = (1e7, 0.0, 0.0)
    s[3] = (-300.0, 2.0, 1.0)
    s[4] = 0.0
    d[5] = 0.0
    d[6] = np.nan
    d[7] = (np.inf, 0.0, 0.0)
    s[8:40] = np.round(s[8:40])
    d[8:40] = np.round(d[8:40]) * 0.0 + (1.0, 0.0, 0.0)
    tree = scenes.random_csg_spec(4, 90)
    specs = [tree]
    chain = []
    for k in range(60):
        chain += [("sphere", 0.3 + 0.01 * k), ("move", -4.0 + 0.15 * k, 0.1 * (k % 7), 0.0)]
    specs.append(chain + [("diff",) if k % 3 else ("blend_union", 0.1) for k in range(59)])
    specs.append(tree + [("flate", 0.1), ("scale", 1.2), ("box", 1.0, 2.0, 0.5), ("blend_diff", 0.2)])
    specs.append(tree + [("ellipsoid", 1.0, 0.5, 0.7), ("union",)])
    specs.append(tree + [("plane", 0.0, 0.0, 1.0), ("inter",)])
    for k, spec in enumerate(specs):
        _same(scenes.build_sdf(spec).program(), s, d)


def test_repeats_share_a_workspace(gpu):
    """Calls of different programs and sizes in turn, and from threads: every
    call's workspace is its own while it runs."""
    from concurrent.futures import ThreadPoolExecutor

    from tangerine_amd import scenes
    jobs = []
    for k, (prims, n) in enumerate([(60, 500), (256, 5000), (20, 64), (120, 2500)] * 2):
        prog = scenes.build_sdf(scenes.random_csg_spec(20 + k, prims)).program()
        s, d = _rays(k, n)
        jobs.append((prog, s, d, _march("tg_raymarch_static", prog, s, d, 100, 1e-3, math.inf, 0)))
    with ThreadPoolExecutor(4) as ex:
        got = list(ex.map(lambda j: _march("tg_raymarch", *j[:3], 100, 1e-3, math.inf, 0), jobs * 3))
    for g, j in zip(got, jobs * 3):
        assert all(np.array_equal(x, y) for x, y in zip(g[:2], j[3][:2]))
