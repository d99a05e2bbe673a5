"""Host point queries staged in pinned memory or device buffers: the same values
on both sides of the line, calls of all sizes one after another in one workspace,
results written over their own points, and several threads at once.
"""

import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def test_staged_queries(gpu):
    from tangerine_amd import _lib, scenes, trace
    prog = scenes.build_sdf(scenes.random_csg_spec(2, 8)).program()
    x = (12.0 * np.random.default_rng(1).random((1000, 3)) - 6.0).astype(np.float32)
    ref, gref = _bits(prog.eval_points(x)), _bits(trace.gradient(prog, x))
    edge_p, edge_g = (16 << 20) // 16, (16 << 20) // 24   # most points / gradients in pinned memory
    for n in (1, 4096, edge_p, 7, edge_p + 1, 1000):
        assert np.array_equal(_bits(prog.eval_points(np.resize(x, (n, 3)))), np.resize(ref, n)), n
    for n in (1, edge_g + 1, 3, edge_g, 1000):
        assert np.array_equal(_bits(trace.gradient(prog, np.resize(x, (n, 3)))), np.resize(gref, (n, 3))), n
    # results over the points themselves
    y = x.copy()
    ptr = y.ctypes.data_as(_lib._fp)
    _lib.check(_lib.load().tg_gradient_points(prog.handle, ptr, 1000, C.c_float(1e-4), 0, ptr, 0), "gradient")
    assert np.array_equal(_bits(y), gref)


def test_staged_queries_of_several_threads(gpu):
    from tangerine_amd import scenes
    prog = scenes.build_sdf(scenes.random_csg_spec(6, 40)).program()
    x = (12.0 * np.random.default_rng(2).random((5000, 3)) - 6.0).astype(np.float32)
    ref = _bits(prog.eval_points(x))
    wrong = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(40):
            a = int(rng.integers(0, 4900))
            n = int(rng.integers(1, 5000 - a))
            if not np.array_equal(_bits(prog.eval_points(x[a:a + n])), ref[a:a + n]):
                wrong.append((k, a, n))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
