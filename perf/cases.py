"""Performance cases: what a program that uses this framework has it do, each
through a public entry point, over the range of sizes that such programs use.

A case is a dict of plain values; `kind` names the path.  Trees are seeded
random CSG trees (sphere, box, torus, cylinder, cone; rotated and translated;
neighbours combined first, in a balanced tree of the six set operators), the
workload of the benchmark and the tests.  Numerics are exact unless a case
says `fast`.

  eval      one distance at one point (a script's `eval` call): pure latency
  points    distances at many points already on the device (sampling for
            training, collision checks)
  gradient  normals at points near the surface, host arrays in and out (mesh
            shading)
  rays      batched ray casts from host arrays (picking, line of sight)
  render    a sphere-traced camera frame with normals, read back
  sodapop   the interactive mesher's job: export, vertex shuffle, normals
  export    a grid export and its mesh, read back
  culled    a certified surrogate-culled export and its mesh, read back
  batch     one batched export of many trees of uneven size, meshes read back
  cloud     a refined point cloud, read back
  fit       a surrogate fitted on the device (forward, backward, Adam)
"""

import math

import numpy as np
import torch

from tangerine_amd import _lib, scenes, trace
from tangerine_amd.batch import Batch
from tangerine_amd.export import Mesher
from tangerine_amd.surrogate import Surrogate

REACH = 4.0      # translations of a tree's primitives
BOUND = 6.0      # half edge of the cube that grids and sample points cover
ROOM = 16        # room a program keeps for a mesh: vertices for each cell of a face
FIELD_FLOPS = 40  # one primitive with its transform, the least a distance costs


def listed():
    return [
        # a script asking for one distance of a small part
        {"name": "eval_one", "kind": "eval", "prims": 3, "fast": False},
        # two million samples of the standard 256-primitive tree, odd count
        {"name": "points_2m", "kind": "points", "prims": 256, "points": 2_000_003, "fast": False},
        # shading normals of a medium mesh
        {"name": "gradient_100k", "kind": "gradient", "prims": 256, "points": 100_003, "fast": False},
        # incoherent ray casts, as a game or a robot program issues them in bulk
        {"name": "rays_50k", "kind": "rays", "prims": 256, "rays": 50_003, "fast": False},
        # the standard frame: 1920x1080, at most 256 steps, normals
        {"name": "render_1080p", "kind": "render", "prims": 256, "width": 1920, "height": 1080, "fast": False},
        # the interactive mesher on a small part at its default density
        {"name": "sodapop_16", "kind": "sodapop", "prims": 16, "density": 20.0, "fast": False},
        # a ragged, non-cubic export in fast numerics
        {"name": "export_ragged", "kind": "export", "prims": 256, "sx": 201, "sy": 150, "sz": 247, "bound": 6.0,
         "fast": True},
        # the headline export
        {"name": "export_1024", "kind": "export", "prims": 2048, "sx": 1024, "sy": 1024, "sz": 1024, "bound": 8.0,
         "fast": False},
        # learned culling with the certificate, half the headline's resolution
        {"name": "culled_512", "kind": "culled", "prims": 2048, "cells": 512, "fast": False},
        # a queue of uneven parts
        {"name": "batch_24", "kind": "batch", "trees": 24, "lo": 8, "hi": 512, "cells": 192, "fast": False},
        # a point cloud with two refinement steps
        {"name": "cloud_120", "kind": "cloud", "prims": 256, "cells": 120, "refine": 2, "fast": False},
        # a short fit: 16 batches of 16384 points, four passes over them
        {"name": "fit_64", "kind": "fit", "prims": 256, "samples": 262_144, "epochs": 4},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["eval", "points", "gradient", "rays", "render", "sodapop", "export", "culled", "batch", "cloud",
                       "fit"])
    case = {"kind": kind, "prims": _log_int(rng, 3, 512), "fast": rng.random() < 0.25}
    if kind == "points":
        case["points"] = _log_int(rng, 100, 2_000_000)
    elif kind == "gradient":
        case["points"] = _log_int(rng, 1, 200_000)
    elif kind == "rays":
        case["rays"] = _log_int(rng, 1, 100_000)
    elif kind == "render":
        case["width"] = _log_int(rng, 64, 1920)
        case["height"] = max(36, int(case["width"] * rng.uniform(0.5, 0.6)))
    elif kind == "sodapop":
        case["prims"] = _log_int(rng, 3, 64)
        case["density"] = round(rng.uniform(8.0, 24.0), 2)
    elif kind == "export":
        case["prims"] = _log_int(rng, 3, 2048)
        case["bound"] = rng.choice([6.0, 8.0])
        base = _log_int(rng, 24, 600)
        for k in ("sx", "sy", "sz"):
            case[k] = max(1, int(base * rng.uniform(0.6, 1.1)))
    elif kind == "culled":
        case["prims"] = _log_int(rng, 16, 2048)
        case["cells"] = _log_int(rng, 64, 512)
    elif kind == "batch":
        del case["prims"]
        case.update(trees=rng.randint(2, 30), lo=4, hi=_log_int(rng, 16, 512), cells=_log_int(rng, 48, 192))
    elif kind == "cloud":
        case["cells"] = _log_int(rng, 16, 160)
        case["refine"] = rng.randint(0, 3)
    elif kind == "fit":
        case["prims"] = _log_int(rng, 16, 512)
        case["samples"] = 16_384 * rng.randint(1, 24)
        case["epochs"] = rng.randint(1, 4)
        del case["fast"]
    return case


# ---- inputs --------------------------------------------------------------------

_OPS = ("union", "diff", "inter", "blend_union", "blend_diff", "blend_inter")


def _f32(v):
    return float(np.float32(v))


def _tree(seed, n):
    """Postfix tokens of a seeded random tree of n primitives."""
    rng = np.random.default_rng(seed)
    kinds = rng.integers(0, 5, n)
    sizes = rng.uniform(0.2, 1.5, (n, 3))
    quats = rng.normal(size=(n, 4))
    quats /= np.linalg.norm(quats, axis=1, keepdims=True)
    moves = rng.uniform(-REACH, REACH, (n, 3))
    cell = np.clip((moves + REACH) / (2 * REACH) * 1023, 0, 1023).astype(np.int64)
    code = np.zeros(n, dtype=np.int64)
    for bit in range(10):
        for axis in range(3):
            code |= ((cell[:, axis] >> bit) & 1) << (3 * bit + axis)
    prims = []
    for i in np.argsort(code, kind="stable"):
        a, b, c = (_f32(v) for v in sizes[i])
        brush = [("sphere", a), ("box", a, b, c), ("torus", a, _f32(0.3 * b)), ("cylinder", a, b), ("cone", a, b)]
        prims.append([brush[kinds[i]], ("rotate", *(_f32(v) for v in quats[i])), ("move", *(_f32(v) for v in moves[i]))])
    out = []

    def rec(lo, hi):
        if hi - lo == 1:
            out.extend(prims[lo])
            return
        mid, m = (lo + hi) // 2, hi - lo
        rec(lo, mid)
        rec(mid, hi)
        p = [1 / 6] * 6 if m <= 4 else [0.35, 0.15, 0, 0.35, 0.15, 0] if m <= 32 else [0.5, 0, 0, 0.5, 0, 0]
        op = _OPS[int(rng.choice(6, p=p))]
        t = _f32(rng.uniform(0.05, 0.3))
        out.append((op, t) if op.startswith("blend") else (op,))

    rec(0, n)
    return out


def _points(seed, n, tree, near):
    """n points: a share `near` around the primitives' surfaces, the rest
    uniform in the cube."""
    rng = np.random.default_rng([seed, 1])
    p = rng.uniform(-BOUND, BOUND, (n, 3))
    brushes = [(t[1], tree[i + 2][1:]) for i, t in enumerate(tree) if t[0] in scenes.BRUSHES]
    at = np.array([b[1] for b in brushes])
    size = np.array([b[0] for b in brushes])
    pick = rng.integers(0, len(brushes), n)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    q = at[pick] + d * (size[pick] + rng.normal(0.0, 0.05, n))[:, None]
    return np.where((rng.random(n) < near)[:, None], q, p).astype(np.float32)


def _rays(seed, n):
    """Starts around the scene, directions towards points inside it."""
    rng = np.random.default_rng([seed, 2])
    s = rng.normal(size=(n, 3))
    s *= 12.0 / np.linalg.norm(s, axis=1, keepdims=True)
    d = rng.uniform(-REACH, REACH, (n, 3)) - s
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return s.astype(np.float32), d.astype(np.float32)


def _grid(cells, bound=BOUND):
    """Origin, step and cells of a grid over the cube (step from its longest axis)."""
    return (_f32(-bound),) * 3, (_f32(2 * bound / max(cells)),) * 3, tuple(cells)


def _cells(case):
    if case["kind"] == "export":
        return (case["sx"], case["sy"], case["sz"])
    if case["kind"] == "sodapop":
        return (int(2 * BOUND * math.floor(case["density"])) + 3,) * 3
    return (case["cells"],) * 3


def _face(cells):
    return (cells[0] * cells[1] + cells[1] * cells[2] + cells[0] * cells[2]) // 3


def _room(cells):
    return ROOM * _face(cells) + 4096


def _pinned(*shape, dtype=torch.float32):
    """A page-locked host array, as a program keeps one for results it reads back."""
    return torch.zeros(shape, dtype=dtype, pin_memory=True).numpy()


def _mesh_buffers(cells):
    n = _room(cells)
    return _pinned(n, 3), _pinned(5 * n // 2, 3, dtype=torch.int32)


def _read_mesh(mesher, buffers):
    """The mesher's mesh into the program's own buffers, as counts and the buffers."""
    v, t = buffers
    nv, nt = mesher.counts()
    if nv > len(v) or nt > len(t):
        raise RuntimeError(f"{nv} vertices and {nt} triangles do not fit")
    _lib.check(mesher.lib.tg_mesher_copy_mesh(mesher.h, v.ctypes.data_as(_lib._fp), t.ctypes.data_as(_lib._u32p)),
               "tg_mesher_copy_mesh")
    return {"counts": np.array([nv, nt]), "vertices": v, "triangles": t}


def _batch_parts(case, seed):
    rng = np.random.default_rng([seed, 3])
    parts = []
    for i in range(case["trees"]):
        n = int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        cells = max(16, int(case["cells"] * (1 / 3, 1 / 2, 2 / 3, 1)[i % 4]))
        parts.append((_tree(seed * 1000 + i, n), cells))
    return parts


def _program(tree):
    return scenes.build_sdf(tree).program()


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "fast": bool(case.get("fast", False))}
    if kind == "batch":
        parts = _batch_parts(case, seed)
        s.update(batch=Batch(), programs=[_program(t) for t, _ in parts], grids=[_grid((c,) * 3) for _, c in parts],
                 buffers=[_mesh_buffers((c,) * 3) for _, c in parts])
        return s
    tree = _tree(seed, case["prims"])
    if kind == "eval":
        node = scenes.build_sdf(tree)
        node.program()
        s.update(node=node, point=tuple(float(v) for v in _points(seed, 1, tree, 0.5)[0]))
        return s
    s["program"] = _program(tree)
    if kind == "points":
        s["xyz"] = torch.from_numpy(_points(seed, case["points"], tree, 0.5)).cuda()
        s["out"] = torch.empty(case["points"], dtype=torch.float32, device="cuda")
    elif kind == "gradient":
        s["xyz"] = _points(seed, case["points"], tree, 1.0)
    elif kind == "rays":
        s["starts"], s["dirs"] = _rays(seed, case["rays"])
    elif kind == "render":
        s["tracer"] = trace.Tracer()
        s["camera"] = trace.look_at(trace.seeded_eye(seed), width=case["width"], height=case["height"])
        n = case["width"] * case["height"]
        s["frame"] = _pinned(n), _pinned(n, 3), _pinned(n, dtype=torch.int32)
    elif kind == "sodapop":
        s["mesher"] = Mesher()
        s["bounds"] = np.array([[-BOUND] * 3, [BOUND] * 3], dtype=np.float32)
        s["buffers"] = _mesh_buffers(_cells(case))
        s["normals"] = _pinned(_room(_cells(case)), 3)
    elif kind == "export":
        s["mesher"] = Mesher()
        s["grid"] = _grid(_cells(case), case["bound"])
        s["buffers"] = _mesh_buffers(_cells(case))
    elif kind == "culled":
        s["mesher"] = Mesher()
        s["grid"] = _grid(_cells(case))
        s["buffers"] = _mesh_buffers(_cells(case))
        s["surrogate"] = Surrogate((-BOUND - 0.25,) * 3, 2 * BOUND + 0.5, seed=seed + 1)
        s["surrogate"].fit(s["program"], samples=131_072, calib_samples=20_000, epochs=8)
    elif kind == "cloud":
        s["mesher"] = Mesher()
        s["step"] = _f32(2 * BOUND / case["cells"])
        s["buffers"] = _mesh_buffers(_cells(case))
    elif kind == "fit":
        s["surrogate"] = Surrogate((-BOUND - 0.25,) * 3, 2 * BOUND + 0.5, seed=seed + 1)
        s["start"] = s["surrogate"].params()
    return s


# ---- one pass --------------------------------------------------------------------

def run(s):
    case, kind, fast = s["case"], s["case"]["kind"], s["fast"]
    if kind == "eval":
        return s["node"].eval(*s["point"], fast=fast)
    if kind == "points":
        _lib.check(_lib.load().tg_eval_points_device(
            s["program"].handle, s["xyz"].data_ptr(), case["points"], s["out"].data_ptr(),
            _lib.TG_FLAG_FAST if fast else 0, torch.cuda.current_stream().cuda_stream), "tg_eval_points_device")
        return s["out"]
    if kind == "gradient":
        return trace.gradient(s["program"], s["xyz"], fast=fast)
    if kind == "rays":
        hit, t, pos = trace.raymarch(s["program"], s["starts"], s["dirs"], fast=fast)
        return {"hit": hit, "t": t, "position": pos}
    if kind == "render":
        s["tracer"].render(s["program"], s["camera"], fast=fast)
        t, normals, steps = s["frame"]
        _lib.check(_lib.load().tg_tracer_copy(s["tracer"].h, t.ctypes.data_as(_lib._fp), normals.ctypes.data_as(_lib._fp),
                                              steps.ctypes.data_as(_lib._u32p)), "tg_tracer_copy")
        return {"t": t, "normals": normals, "steps": steps}
    if kind == "sodapop":
        s["mesher"].export_sodapop(s["program"], s["bounds"], density=case["density"], fast=fast)
        out = _read_mesh(s["mesher"], s["buffers"])
        _lib.check(_lib.load().tg_mesher_copy_normals(s["mesher"].h, s["normals"].ctypes.data_as(_lib._fp)),
                   "tg_mesher_copy_normals")
        out["normals"] = s["normals"]
        return out
    if kind == "export":
        s["mesher"].export(s["program"], *s["grid"], fast=fast)
        return _read_mesh(s["mesher"], s["buffers"])
    if kind == "culled":
        s["mesher"].export_culled(s["program"], s["surrogate"], *s["grid"], fast=fast)
        return _read_mesh(s["mesher"], s["buffers"])
    if kind == "batch":
        s["batch"].export(s["programs"], s["grids"], fast=fast)
        parts = [_read_mesh(s["batch"].mesher(i), b) for i, b in enumerate(s["buffers"])]
        return {"counts": np.array([p["counts"] for p in parts]), "vertices": [p["vertices"] for p in parts],
                "triangles": [p["triangles"] for p in parts]}
    if kind == "cloud":
        s["mesher"].export_points(s["program"], (-BOUND,) * 3, (BOUND,) * 3, s["step"], case["refine"], fast=fast)
        return _read_mesh(s["mesher"], s["buffers"])
    s["surrogate"].set_params(*s["start"])
    s["surrogate"].fit(s["program"], samples=case["samples"], calib_samples=20_000, epochs=case["epochs"])
    return {"params": s["surrogate"].params()[0], "loss": s["surrogate"].loss_log()}


def work(case):
    kind = case["kind"]
    records = 64 * (2 * case.get("prims", 0))
    if kind == "eval":
        return {"bytes": records + 16, "flops": FIELD_FLOPS}
    if kind == "points":
        return {"bytes": records + 16 * case["points"], "flops": FIELD_FLOPS * case["points"]}
    if kind == "gradient":
        return {"bytes": records + 24 * case["points"], "flops": 4 * FIELD_FLOPS * case["points"]}
    if kind == "rays":  # about ten steps to the surface
        return {"bytes": records + 41 * case["rays"], "flops": 10 * FIELD_FLOPS * case["rays"]}
    if kind == "render":  # the same, and six taps for a normal
        n = case["width"] * case["height"]
        return {"bytes": records + 20 * n, "flops": 16 * FIELD_FLOPS * n}
    if kind == "cloud":
        n = case["cells"] ** 3
        kept = 12 * case["cells"] ** 2
        return {"bytes": records + 12 * kept, "flops": FIELD_FLOPS * (n + 5 * kept * case["refine"])}
    if kind == "fit":
        steps = case["samples"] // 16_384 * case["epochs"]
        per_point = 3 * 2 * (96 * 64 + 64 * 64 + 64)
        return {"bytes": records + 16 * case["samples"] + 4 * 10_433, "flops": steps * 16_384 * per_point}
    if kind == "batch":
        sizes = [max(16, int(case["cells"] * f)) for f in (1 / 3, 1 / 2, 2 / 3, 1)]
        per = sum(_export_bytes((c, c, c)) for c in sizes) / 4
        cells = sum((c + 1) ** 3 for c in sizes) / 4
        return {"bytes": case["trees"] * per, "flops": case["trees"] * FIELD_FLOPS * cells}
    cells = _cells(case)
    if kind == "culled":
        n = 6 * _face(cells)  # bricks' worth of samples next to the surface
        return {"bytes": records + 4 * 8 * n + _mesh_bytes(cells), "flops": FIELD_FLOPS * 8 * n}
    samples = (cells[0] + 1) * (cells[1] + 1) * (cells[2] + 1)
    normals = 12 * 7 * _face(cells) if kind == "sodapop" else 0
    return {"bytes": records + _export_bytes(cells) + normals, "flops": FIELD_FLOPS * (samples + normals // 3)}


def _mesh_bytes(cells):
    """About seven vertices for each cell of a face, two triangles a vertex."""
    return 7 * _face(cells) * 36


def _export_bytes(cells):
    return 4 * (cells[0] + 1) * (cells[1] + 1) * (cells[2] + 1) + _mesh_bytes(cells)


# ---- the same in 64 bits ------------------------------------------------------------

class _Field:
    """A tree's distance in float64 with torch: every primitive of a kind at
    once, then the operators in postfix order."""

    def __init__(self, tree):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dev, self.groups, self.ops = dev, {}, []
        count = 0
        for i, t in enumerate(tree):
            if t[0] in ("rotate", "move"):
                continue
            if t[0] in _OPS:
                self.ops.append(t)
                continue
            self.groups.setdefault(t[0], []).append((count, t[1:], tree[i + 1][1:], tree[i + 2][1:]))
            self.ops.append(count)
            count += 1
        self.count = count
        for kind, rows in self.groups.items():
            q = torch.tensor([r[2] for r in rows], dtype=torch.float64, device=dev)
            q = q / q.norm(dim=1, keepdim=True)
            x, y, z, w = q.unbind(1)
            m = [1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                 2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                 2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]
            par = torch.zeros((len(rows), 3), dtype=torch.float64, device=dev)
            for k, r in enumerate(rows):
                par[k, : len(r[1])] = torch.tensor(r[1], dtype=torch.float64)
            at = torch.tensor([r[3] for r in rows], dtype=torch.float64, device=dev)
            idx = torch.tensor([r[0] for r in rows], device=dev)
            self.groups[kind] = (idx, [v[:, None] for v in m], at, par)

    def _brush(self, kind, x, y, z, par):
        a, b, c = (par[:, k, None] for k in range(3))
        if kind == "sphere":
            return (x * x + y * y + z * z).sqrt() - a
        if kind == "box":
            x, y, z = x.abs() - a, y.abs() - b, z.abs() - c
            out = (x.clamp(min=0) ** 2 + y.clamp(min=0) ** 2 + z.clamp(min=0) ** 2).sqrt()
            return out + torch.maximum(torch.maximum(x, y), z).clamp(max=0)
        r = (x * x + y * y).sqrt()
        if kind == "torus":
            return ((r - a) ** 2 + z * z).sqrt() - b
        if kind == "cylinder":
            r, z = r - a, z.abs() - b
            return torch.maximum(r, z).clamp(max=0) + (r.clamp(min=0) ** 2 + z.clamp(min=0) ** 2).sqrt()
        # cone of base radius a and height b about the origin, apex up: the
        # nearest point of its slope and of its base
        w = z - 0.5 * b
        t = ((r * a - w * b) / (a * a + b * b)).clamp(0, 1)
        u = (r / a).clamp(0, 1)
        d = torch.minimum((r - a * t) ** 2 + (w + b * t) ** 2, (r - a * u) ** 2 + (w + b) ** 2)
        s = torch.maximum(r * b + w * a, -(w + b))
        return d.sqrt() * torch.sign(s)

    def _chunk(self, p):
        d = torch.empty((self.count, p.shape[0]), dtype=torch.float64, device=self.dev)
        for kind, (idx, m, at, par) in self.groups.items():
            x, y, z = (p[:, k][None] - at[:, k, None] for k in range(3))
            d[idx] = self._brush(kind, m[0] * x + m[3] * y + m[6] * z, m[1] * x + m[4] * y + m[7] * z,
                                 m[2] * x + m[5] * y + m[8] * z, par)
        stack = []
        for t in self.ops:
            if isinstance(t, int):
                stack.append(d[t])
                continue
            b, a = stack.pop(), stack.pop()
            if t[0].endswith("diff"):
                b = -b
            v = torch.minimum(a, b) if t[0].endswith("union") else torch.maximum(a, b)
            if len(t) > 1:
                h = (t[1] - (a - b).abs()).clamp(min=0) ** 2 * (0.25 / t[1])
                v = v - h if t[0].endswith("union") else v + h
            stack.append(v)
        return stack[0]

    def __call__(self, p):
        step = max(1024, (1 << 25) // self.count)
        parts = [self._chunk(p[i:i + step]) for i in range(0, p.shape[0], step)]
        return torch.cat(parts) if parts else torch.empty(0, dtype=torch.float64, device=self.dev)

    def gradient(self, p, h=1e-4):
        o = torch.tensor([[1, -1, -1], [-1, -1, 1], [-1, 1, -1], [1, 1, 1]], dtype=torch.float64, device=self.dev)
        g = sum(self(p + h * o[k])[:, None] * o[k] for k in range(4))
        return g / g.norm(dim=1, keepdim=True)

    def axis(self, lo, step, n):
        """Grid samples along one axis, as single precision places them."""
        v = np.float32(lo) + np.arange(n, dtype=np.float32) * np.float32(step)
        return torch.from_numpy(v).to(self.dev, torch.float64)


def _in_room(v, cells):
    """Vertices as a program's buffer holds them: zeros behind the last."""
    out = torch.zeros((_room(cells), 3), dtype=torch.float64, device=v.device)
    out[: len(v)] = v[: len(out)]
    return out


def _mesh_vertices(field, origin, step, cells):
    """Naive surface nets' vertices of a grid, in raster order."""
    x, y, z = (field.axis(origin[k], step[k], cells[k] + 1) for k in range(3))
    p = torch.stack(torch.meshgrid(z, y, x, indexing="ij"), -1).flip(-1).reshape(-1, 3)
    d = field(p).reshape(cells[2] + 1, cells[1] + 1, cells[0] + 1)
    del p
    sx, sy, sz = cells
    pos = d >= 0
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    part = [pos[c:c + sz, b:b + sy, a:a + sx] for a, b, c in corner]
    every, some = part[0].clone(), part[0].clone()
    for q in part[1:]:
        every &= q
        some |= q
    k, j, i = torch.nonzero(some & ~every, as_tuple=True)
    s = [d[k + c, j + b, i + a] for a, b, c in corner]
    total = torch.zeros((len(i), 3), dtype=torch.float64, device=d.device)
    n = torch.zeros(len(i), dtype=torch.float64, device=d.device)
    for e, f in ((0, 1), (1, 2), (2, 3), (3, 0), (4, 5), (5, 6), (6, 7), (7, 4), (0, 4), (1, 5), (2, 6), (3, 7)):
        cross = ((s[e] >= 0) != (s[f] >= 0)).double()
        t = torch.where(cross > 0, -s[e] / (s[f] - s[e]), torch.zeros_like(s[e]))
        for ax in range(3):
            total[:, ax] += cross * (corner[e][ax] + t * (corner[f][ax] - corner[e][ax]))
        n += cross
    base = torch.stack([i, j, k], 1).double()
    o, h = (torch.tensor(v, dtype=torch.float64, device=d.device) for v in (origin, step))
    return _in_room(o + (base + total / n[:, None]) * h, cells)


def _march(field, starts, dirs, max_steps=100, eps=1e-3):
    o = torch.from_numpy(starts).to(field.dev, torch.float64)
    v = torch.from_numpy(dirs).to(field.dev, torch.float64)
    v = v / v.norm(dim=1, keepdim=True)
    t = torch.zeros(len(o), dtype=torch.float64, device=field.dev)
    hit = torch.zeros(len(o), dtype=torch.bool, device=field.dev)
    live = torch.arange(len(o), device=field.dev)
    for _ in range(max_steps):
        d = field(o[live] + v[live] * t[live, None])
        on = d <= float(np.float32(eps))
        hit[live[on]] = True
        live, d = live[~on], d[~on]
        if not len(live):
            break
        t[live] += d
    return {"hit": None, "t": torch.where(hit, t, torch.full_like(t, math.inf)), "position": o + v * t[:, None]}


def _cloud(field, case):
    step = np.float32(2 * BOUND / case["cells"])
    n = int(math.ceil(float((np.float32(BOUND) - np.float32(-BOUND)) / step)))
    half = float(step) / 2
    x = torch.from_numpy((np.arange(n, dtype=np.float32) * step + np.float32(-BOUND)) + step / np.float32(2))
    x = x.to(field.dev, torch.float64)
    p = torch.stack(torch.meshgrid(x, x, x, indexing="ij"), -1).flip(-1).reshape(-1, 3)
    far = half * math.sqrt(3)
    p = p[field(p).abs() < far]
    c = p.clone()
    for _ in range(case["refine"]):
        c = c - field.gradient(c) * field(c)[:, None]
    c = torch.maximum(torch.minimum(c, p + half), p - half)
    return torch.where(((c - p).norm(dim=1) <= far)[:, None], c, p)


def exact(case, seed):
    kind = case["kind"]
    # a frame's grazing rays hit or miss by their last bit, a sodapop mesh is
    # shuffled by the C++ library's own algorithm, a fit draws its samples
    # on the device, and in fast numerics a cube that the surface only touches
    # may come or go, which moves every vertex behind it
    if kind in ("render", "sodapop", "fit") or (case["fast"] and kind in ("export", "culled", "batch", "cloud")):
        return None
    if kind == "batch":
        parts = _batch_parts(case, seed)
        if sum(sum(t[0] in scenes.BRUSHES for t in tree) * (c + 1) ** 3 for tree, c in parts) > 6e9:
            return None
        return {"counts": None, "vertices": [_mesh_vertices(_Field(tree), *_grid((c,) * 3)) for tree, c in parts],
                "triangles": [None] * len(parts)}
    tree = _tree(seed, case["prims"])
    if kind in ("export", "culled"):
        cells = _cells(case)
        if case["prims"] * (cells[0] + 1) * (cells[1] + 1) * (cells[2] + 1) > 6e9:
            return None
        grid = _grid(cells, case.get("bound", BOUND))
        return {"counts": None, "vertices": _mesh_vertices(_Field(tree), *grid), "triangles": None}
    field = _Field(tree)
    if kind == "rays":
        return _march(field, *_rays(seed, case["rays"]))
    if kind == "cloud":
        return {"counts": None, "vertices": _in_room(_cloud(field, case), _cells(case)), "triangles": None}
    n = 1 if kind == "eval" else case["points"]
    near = 1.0 if kind == "gradient" else 0.5
    p = torch.from_numpy(_points(seed, n, tree, near)).to(field.dev, torch.float64)
    if kind == "eval":
        return float(field(p)[0])
    return field(p) if kind == "points" else field.gradient(p)
