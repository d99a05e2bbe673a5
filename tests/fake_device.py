"""Runs a script against libtangerine_gpu.so with tests/fake_hip.cpp in the HIP
runtime's place: the library's host code without a device."""

import atexit
import functools
import shutil
import subprocess
import sys
import tempfile
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
fake = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
fake.fake_launches.restype = C.c_char_p
fake.fake_limit.argtypes = [C.c_size_t]
for name in ("used", "peak", "mallocs"):
    getattr(fake, "fake_" + name).restype = C.c_size_t
fake.fake_pending.restype = C.c_long
import numpy as np
from tangerine_amd import _lib, scenes
lib = _lib.load()
_lib.check(lib.tg_device_init(0), "tg_device_init")

def launches():
    "Kernels launched since the last call: (name, workgroups, threads, LDS bytes)."
    out = []
    for line in fake.fake_launches().decode().splitlines():
        name, grid, block, lds = line.rsplit(" ", 3)
        out.append((name, int(grid), int(block), int(lds)))
    return out

def ran(kernel, calls):
    return any(kernel in c[0] for c in calls)

def program(prims, seed=1):
    return scenes.build_sdf(scenes.random_csg_spec(seed, prims)).program()
"""


@functools.lru_cache(maxsize=1)
def _fake_lib():
    from tangerine_amd.build import HIPCC
    out = Path(tempfile.mkdtemp(prefix="fake_hip_")) / "libfake_hip.so"
    atexit.register(shutil.rmtree, out.parent, True)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(out),
                    str(ROOT / "tests" / "fake_hip.cpp")], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    return out


def run(script, timeout=240):
    """The script's stdout; fails the test with its stderr."""
    head = PRELUDE.format(root=str(ROOT), lib=str(_fake_lib()))
    p = subprocess.run([sys.executable, "-c", head + script], capture_output=True, text=True, timeout=timeout, cwd=ROOT)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout
