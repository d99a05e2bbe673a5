"""Frames of programs that no cell prunes (an ellipsoid) or hardly any (wide blends),
and unpruned renders: small ones with groups of lanes, larger ones in passes.  Image,
step counts and counters equal the same frame's in one pass.
"""

import numpy as np
import pytest

from tests.test_gpu_trace_groups import _frame

pytestmark = pytest.mark.gpu


def _spec(kind, prims):
    from tangerine_amd import scenes
    spec = scenes.random_csg_spec(31, prims)
    if kind == "ellipsoid":
        at = next(i for i, t in enumerate(spec) if t[0] in scenes.PRIMITIVES)
        return spec[:at] + [("ellipsoid", 0.5, 0.7, 0.9)] + spec[at + 1:]
    return [("blend_union", 2.0) if t[0] in scenes.SET_OPS else t for t in spec]


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("kind", ["ellipsoid", "blends"])
@pytest.mark.parametrize("prims,width,height", [(30, 97, 55), (200, 160, 90), (30, 701, 401)])
def test_same_frame(gpu, kind, prims, width, height, fast):
    from tangerine_amd import scenes, trace
    prog = scenes.build_sdf(_spec(kind, prims)).program()
    cam = trace.look_at((9.0, 6.0, 5.0), (0, 0, 0), (0, 0, 1), 60.0, width, height)
    ref_st, ref = _frame(prog, cam, True, 256, 1e-3, fast, 40.0)
    st, got = _frame(prog, cam, False, 256, 1e-3, fast, 40.0)
    tr = trace.Tracer()
    tr.render(prog, cam, 256, 1e-4, 40.0, 1e-3, fast=fast, prune=False)
    whole = tr.image()
    tr.close()
    for a, b, c in zip(got, ref, whole):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert np.array_equal(np.array(c).view(np.uint32), b.view(np.uint32))
    assert st["hits"] == ref_st["hits"] and st["evaluations"] == ref_st["evaluations"]
    assert 0 < st["hits"] < width * height
