"""Frames whose long marches go on in groups of lanes, against the same frames in
one pass: image, step counts and counters are equal, for programs that groups of 16
lanes hold, that need a wave to a ray, and that are longer than a wave holds; for
frames smaller than a wave's tile; with and without normals; at the fewest steps
that go this way and next to them.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _frame(prog, cam, one_pass, steps, h, fast, far):
    from tangerine_amd import trace
    tr = trace.Tracer()
    if one_pass:
        tr.set_passes(0, 0, 1)
    st = tr.render(prog, cam, steps, 1e-4, far, h, fast=fast)
    out = [np.array(a) for a in tr.image()]
    tr.close()
    return st, out


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("prims,width,height,steps,h,far", [
    (1, 5, 3, 256, 1e-3, 40.0), (20, 97, 55, 256, 1e-3, 40.0), (128, 97, 55, 17, 1e-3, 40.0), (129, 97, 55, 256, 0.0, 40.0),
    (300, 160, 90, 256, 1e-3, 40.0), (300, 97, 55, 16, 1e-3, 40.0), (300, 97, 55, 49, 0.3, 1e6), (300, 64, 36, 300, 1e-3, 5.0),
    (4100, 33, 17, 64, 1e-3, 40.0)])
def test_groups_give_the_same_frame(gpu, prims, width, height, steps, h, far, fast):
    from tangerine_amd import scenes, trace
    prog = scenes.build_sdf(scenes.random_csg_spec(21, prims)).program()
    for eye in [(9.0, 6.0, 5.0), (0.4, -0.3, 7.0)]:
        cam = trace.look_at(eye, (0, 0, 0), (0, 0, 1), 60.0, width, height)
        ref_st, ref = _frame(prog, cam, True, steps, h, fast, far)
        st, got = _frame(prog, cam, False, steps, h, fast, far)
        for a, b in zip(got, ref):
            assert a.dtype == b.dtype and np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert st["hits"] == ref_st["hits"] and st["evaluations"] == ref_st["evaluations"]
