"""Few points and gradients with the program split over workgroups, and many with
one or two points or taps to a lane: the same values as the oracle, bit for bit.

Sizes on both sides of every line of the dispatch, and remainders of 64 points,
16 points and two points a lane; trees of one treelet (not split), two and more
stages, and one deep chain.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def _points(n, seed):
    rng = np.random.default_rng(seed)
    x = (12.0 * rng.random((n, 3)) - 6.0).astype(np.float32)
    x[:: max(1, n // 7)] *= np.float32(50.0)
    return x


@pytest.mark.parametrize("prims", [3, 16, 17, 33, 48, 256, 700])
def test_points_same_at_every_count(gpu, oracle, prims):
    from tangerine_amd import scenes
    node = scenes.build_sdf(scenes.random_csg_spec(prims, prims))
    prog, words = node.program(), node.compile()
    x = _points(4099, prims)
    ref = _bits(oracle.interp_words(words, x))
    for n in (1, 63, 64, 65, 4099):
        assert np.array_equal(_bits(prog.eval_points(x[:n])), ref[:n]), n
    # a million and a half and one: lane-strided pairs, whole program
    for n in (32768, 32769, 131072, 131073, 1500001):
        big = np.resize(x, (n, 3))
        assert np.array_equal(_bits(prog.eval_points(big)), np.resize(ref, n)), n


@pytest.mark.parametrize("central", [False, True])
@pytest.mark.parametrize("prims", [3, 17, 256])
def test_gradients_same_at_every_count(gpu, prims, central):
    from tangerine_amd import scenes, trace
    prog = scenes.build_sdf(scenes.random_csg_spec(prims + 1, prims)).program()
    x = _points(515, prims + 2)
    x[3] = 0.0
    many = trace.gradient(prog, np.resize(x, (150001, 3)), central=central)  # two taps to a lane
    ref = _bits(many[:515])
    assert np.array_equal(_bits(many), np.resize(ref, (150001, 3)))
    for n in (1, 15, 16, 17, 515):  # split (one tap to a lane for a single treelet)
        assert np.array_equal(_bits(trace.gradient(prog, x[:n], central=central)), ref[:n]), n
    for n in (4096, 4097, 16384, 16385):
        got = trace.gradient(prog, np.resize(x, (n, 3)), central=central)
        assert np.array_equal(_bits(got), np.resize(ref, (n, 3))), n


def test_gradients_match_oracle(gpu, oracle):
    from tangerine_amd import scenes, trace
    node = scenes.build_sdf(scenes.random_csg_spec(5, 64))
    x = _points(300, 9)
    ref = oracle.gradient_tetra(node.compile(), x)
    assert np.array_equal(_bits(trace.gradient(node.program(), x)), _bits(ref))


def test_points_split_under_capture(gpu):
    """The asynchronous call records into a graph; every replay gives the values."""
    import ctypes as C

    from tangerine_amd import _lib, scenes
    prog = scenes.build_sdf(scenes.random_csg_spec(4, 256)).program()
    x = _points(1000, 3)
    ref = _bits(prog.eval_points(x))
    lib = _lib.load()
    hip = lambda name, *args: _check_hip(name, getattr(lib, name)(*args))  # the library's own runtime

    def _check_hip(name, rc):
        assert rc == 0, (name, rc)

    dx, do, stream, graph, run = (C.c_void_p() for _ in range(5))
    hip("hipMalloc", C.byref(dx), C.c_size_t(x.nbytes))
    hip("hipMalloc", C.byref(do), C.c_size_t(4000))
    hip("hipMemcpy", dx, x.ctypes.data_as(C.c_void_p), C.c_size_t(x.nbytes), 1)
    hip("hipStreamCreate", C.byref(stream))
    hip("hipStreamBeginCapture", stream, 2)
    _lib.check(lib.tg_eval_points_device(prog.handle, dx, 1000, do, 0, stream), "points")
    hip("hipStreamEndCapture", stream, C.byref(graph))
    hip("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
    for _ in range(3):
        out = np.zeros(1000, np.float32)
        hip("hipMemcpy", do, out.ctypes.data_as(C.c_void_p), C.c_size_t(4000), 1)
        hip("hipGraphLaunch", run, stream)
        hip("hipStreamSynchronize", stream)
        hip("hipMemcpy", out.ctypes.data_as(C.c_void_p), do, C.c_size_t(4000), 2)
        assert np.array_equal(_bits(out), ref)
    hip("hipGraphExecDestroy", run)
    hip("hipGraphDestroy", graph)
    hip("hipStreamDestroy", stream)
    hip("hipFree", dx)
    hip("hipFree", do)
