"""The work that performance is judged on: shadow DAG builds and lookups through the public entry
points of cpvs_amd, from single small maps to the 8192^2 map and the tiled map's tiles.

A case is a dict of plain values; ``listed()`` gives the fixed ones and ``draw(rng)`` more of the
same ranges.  ``prepare`` makes what a program holds before the call (depth maps and query points
in device memory, built containers, DAG sets or servers), ``run`` is one pass and returns its
outputs as torch views of device buffers.  Maps and points come from torch's generators, with
the shape of the synthetic inputs of bench.py: a tilted plane, optional four-octave value noise and
boxes in front of it; points on the surface, near it, or uniform in the light's volume.
"""
import ctypes
import math
import random

import numpy as np
import torch

import cpvs_amd as cp
from cpvs_amd import _lib


def listed():
    return [
        # The smallest map of the many-maps configuration, built alone: launches and readbacks count.
        {"name": "build_256", "kind": "build", "N": 256, "boxes": 2, "noise": True},
        # The 1024^2 configuration: plane and 32 boxes, without noise.
        {"name": "build_1024", "kind": "build", "N": 1024, "boxes": 32, "noise": False},
        # The headline map.
        {"name": "build_8192", "kind": "build", "N": 8192, "boxes": 512, "noise": True},
        # One xy tile of the 65536^2 tiled map: one pyramid, a DAG for each of its 8 z-tiles, built one
        # after another as the reference's loop does.
        {"name": "tile_8192_z8", "kind": "tile", "N": 8192, "boxes": 256, "T": 8},
        # Many maps of log-uniform size in one batched call.
        {"name": "batch_32_maps", "kind": "batch", "maps": 32, "kmin": 8, "kmax": 12, "mix": 3},
        # One frame with a moving light, as the reference runs it: the shadow map as an image in host
        # memory, pyramid, DAG, container, and the visibility of a G-buffer in world space.
        {"name": "frame_1024_host", "kind": "frame", "N": 1024, "boxes": 32, "host": True, "W": 1920, "H": 1080},
        # The smallest lookup request of the serving mix.
        {"name": "lookup_1k", "kind": "lookup", "N": 1024, "boxes": 32, "points": "uniform", "count": 1000, "stride": 3,
         "matrix": True},
        # The headline lookups: two points for each pixel of a 3840 x 2160 G-buffer.
        {"name": "lookup_gbuffer_4k", "kind": "lookup", "N": 8192, "boxes": 512, "points": "gbuffer", "count": 16588800,
         "stride": 4, "matrix": False},
        # Random points over a container of 4 x 4 x 4 DAGs (a tiled map of 4096^2).
        {"name": "tiled_lookup_4m", "kind": "tiled", "N": 1024, "L": 4, "boxes": 32, "count": 4194301},
        # Filtered shadows of a full-HD frame in world space.
        {"name": "pcf3_1080p", "kind": "pcf", "N": 4096, "boxes": 512, "f": 3, "W": 1920, "H": 1080},
        # Queries over many DAGs in one launch, DAG i mod n for query i, with 4-level top tables.
        {"name": "dagset_48", "kind": "dagset", "dags": 48, "kmin": 8, "kmax": 11, "mix": 5, "count": 6291449, "ids": False,
         "top": 4},
        # A burst of a server's mix: builds and lookups on resident DAGs submitted together.
        {"name": "serve_burst", "kind": "serve", "resident": 8, "builds": 4, "lookups": 24, "kmin": 9, "kmax": 11, "mix": 7},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["build", "build", "tile", "batch", "frame", "lookup", "lookup", "tiled", "pcf", "dagset", "serve"])
    mix = rng.randrange(1 << 20)

    def boxes(N):  # the density of the fixed maps, a quarter of it to twice it
        return max(1, int(32 * (N / 1024) ** 2 * 2.0 ** rng.uniform(-3, 1)))

    if kind == "build":
        N = 1 << rng.randint(8, 13)
        return {"kind": kind, "N": N, "boxes": boxes(N), "noise": rng.random() < 0.7}
    if kind == "tile":
        N = 1 << rng.randint(10, 12)
        return {"kind": kind, "N": N, "boxes": boxes(N), "T": 1 << rng.randint(1, 3)}
    if kind == "batch":
        return {"kind": kind, "maps": _log_int(rng, 4, 32), "kmin": 8, "kmax": rng.randint(9, 12), "mix": mix}
    if kind == "frame":
        N = 1 << rng.randint(9, 11)
        return {"kind": kind, "N": N, "boxes": boxes(N), "host": rng.random() < 0.5, "W": rng.randint(320, 1920),
                "H": rng.randint(240, 1080)}
    if kind == "lookup":
        N = 1 << rng.randint(8, 13)
        return {"kind": kind, "N": N, "boxes": boxes(N), "points": rng.choice(["uniform", "gbuffer"]),
                "count": _log_int(rng, 1000, 16500000), "stride": rng.choice([3, 4]), "matrix": rng.random() < 0.5}
    if kind == "tiled":
        L = rng.choice([2, 4])
        N = 1 << rng.randint(8, 10)
        return {"kind": kind, "N": N, "L": L, "boxes": boxes(N), "count": _log_int(rng, 1000, 8000000)}
    if kind == "pcf":
        N = 1 << rng.randint(9, 12)
        return {"kind": kind, "N": N, "boxes": boxes(N), "f": rng.randint(2, 5), "W": rng.randint(320, 1920),
                "H": rng.randint(240, 1080)}
    if kind == "dagset":
        return {"kind": kind, "dags": _log_int(rng, 3, 64), "kmin": 8, "kmax": rng.randint(9, 11), "mix": mix,
                "count": _log_int(rng, 10000, 6000000), "ids": rng.random() < 0.5, "top": rng.choice([0, 4])}
    return {"kind": "serve", "resident": rng.randint(2, 8), "builds": rng.randint(1, 4), "lookups": rng.randint(4, 32),
            "kmin": 9, "kmax": rng.randint(10, 11), "mix": mix}


# ---- inputs ----------------------------------------------------------------------------------


def _rng(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _noise_octave(u, v, n, g):
    """Value noise: an (n+1)^2 lattice of U[0,1) values, smoothstep-bilinear at v x u in [0, 1]."""
    lat = torch.rand(n + 1, n + 1, generator=g, device="cuda")

    def cell(x):
        i = (x * n).floor().clamp_(max=n - 1).long()
        t = x * n - i
        return i, t * t * (3 - 2 * t)

    (i, t), (j, r) = cell(u), cell(v)
    rows = lat[j] + (lat[j + 1] - lat[j]) * r[:, None]
    a = rows[:, i]
    return a.add_((rows[:, i + 1] - a).mul_(t[None, :]))


def _depth(N, boxes, noise, seed, salt, of=1):
    """An N x N float32 light-space depth map in device memory; with of > 1 one tile of a map of
    of x of tiles (plane and noise span the whole map)."""
    g = _rng(seed, salt)
    r = random.Random((int(seed) * 1000003 + salt) ^ 0x5EED)
    x = (torch.arange(N, device="cuda", dtype=torch.float32) + 0.5) / N
    u, v = (x + r.randrange(of)) / of, (x + r.randrange(of)) / of
    d = (0.6 + 0.1 * u)[None, :].repeat(N, 1)
    if noise:
        for n, w in ((8, 1.0), (16, 0.5), (32, 0.25), (64, 0.125)):
            d.add_(_noise_octave(u, v, n, g).sub_(0.5), alpha=0.05 * w / 1.875)
    d.clamp_(0.0, 1.0)
    for _ in range(boxes):
        s = min(r.randint(16, 128), N)
        x, y, z = r.randint(0, N - s), r.randint(0, N - s), r.uniform(0.1, 0.5)
        d[y:y + s, x:x + s].clamp_(max=z)
    return d


def _uniform(count, stride, seed, salt):
    p = torch.rand(count, stride, generator=_rng(seed, salt), device="cuda").mul_(2.0).sub_(1.0)
    if stride == 4:
        p[:, 3] = 1.0
    return p


def _gbuffer(depth, W, H, both, seed, salt):
    """NDC points (float4) of a W x H image over the map: each pixel's surface point, moved by up to
    two voxels in z; with `both`, the surface point itself as well."""
    N = depth.shape[0]
    u = (torch.arange(W, device="cuda", dtype=torch.float32) + 0.5) / W
    v = (torch.arange(H, device="cuda", dtype=torch.float32) + 0.5) / H
    z = depth[(v * N).long().clamp_(max=N - 1)][:, (u * N).long().clamp_(max=N - 1)]
    jit = (torch.rand(H, W, generator=_rng(seed, salt), device="cuda") * 2 - 1) * (2.0 / N)
    near = (z + jit).clamp_(0.0, 1.0)
    k = 2 if both else 1
    p = torch.ones(H, W, k, 4, device="cuda")
    p[..., 0] = (2 * u - 1)[None, :, None]
    p[..., 1] = (2 * v - 1)[:, None, None]
    if both:
        p[:, :, 0, 2] = 2 * z - 1
    p[:, :, k - 1, 2] = 2 * near - 1
    return p.reshape(-1, 4)


def _light(seed):
    """An orthographic light: (lightViewProj, its inverse), the world a rotated 40-unit box."""
    r = random.Random(int(seed) ^ 0x11617)
    a, b = r.uniform(0.2, 1.2), r.uniform(0.0, 6.2)
    rx = np.array([[1, 0, 0], [0, math.cos(a), -math.sin(a)], [0, math.sin(a), math.cos(a)]])
    rz = np.array([[math.cos(b), -math.sin(b), 0], [math.sin(b), math.cos(b), 0], [0, 0, 1]])
    m = np.eye(4)
    m[:3, :3] = (rx @ rz) / 20.0
    m[:3, 3] = [r.uniform(-0.1, 0.1) for _ in range(3)]
    return m.astype(np.float32), np.linalg.inv(m)


def _to_world(ndc, inverse):
    inv = torch.tensor(inverse, device="cuda", dtype=torch.float32)
    p = ndc.clone()
    p[:, :3] = ndc[:, :3] @ inv[:3, :3].T.contiguous() + inv[:3, 3]
    return p


def _sizes(case, n, salt=0):
    r = random.Random(case["mix"] * 31 + salt)
    s = [1 << r.randint(case["kmin"], case["kmax"]) for _ in range(n)]
    s[0] = 1 << case["kmax"]
    return s


def _boxes_of(N):
    return max(1, (32 * N * N) // (1024 * 1024))


# ---- device buffers --------------------------------------------------------------------------


class _View:
    """Device memory as the array interface that torch reads; keeps its owner alive."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False), "version": 2}


def _tensor(a):
    return torch.as_tensor(_View(a.ptr.value, a.shape, a.dtype.str, a), device="cuda")


def _array(t):
    """A torch tensor's values in a DeviceArray."""
    t = t.contiguous()
    a = cp.DeviceArray(tuple(t.shape), str(t.dtype).replace("torch.", ""))
    if t.numel():
        _tensor(a).copy_(t)
        torch.cuda.synchronize()  # the library works on its own stream
    return a


def _word_room(N):
    """Words that the outputs have room for per DAG of an N x N map (these maps need fewer)."""
    return max(4096, N * N // 6)


def _keep(state, handles, rooms):
    """Copies the DAGs' words into the program's own buffer, each DAG at its own place in it (how many
    there are follows from the map, the outputs' shapes do not).  Returns it and the word counts."""
    buf, at, counts = state["words"], 0, []
    for h, room in zip(handles, rooms):
        n, p = ctypes.c_uint64(), ctypes.c_void_p()
        _lib.call("cpvs_dag_info", h, None, ctypes.byref(n), None)
        _lib.call("cpvs_dag_device_words", h, ctypes.byref(p))
        _lib.call("cpvs_memcpy_d2d", buf.ctx.handle, ctypes.c_void_p(buf.ptr.value + 4 * at), p, 4 * min(n.value, room), None)
        counts.append(n.value)
        at += room
    return [_tensor(buf), np.array(counts, np.int64)]


def _room(state, rooms):
    state["rooms"] = rooms
    state["words"] = _array(torch.zeros(sum(rooms), dtype=torch.int32, device="cuda"))


def _shadow(depth):
    mm = cp.MinMaxHierarchy(_array(depth))
    sh = cp.CompressedShadow.create(mm)
    mm.close()
    return sh


def _container(depth):
    c = cp.CompressedShadowContainer(_shadow(depth))
    c.moveToGPU()
    return c


# ---- a case ----------------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind in ("build", "tile"):
        s["depth"] = _array(_depth(case["N"], case["boxes"], case.get("noise", True), seed, 1, case.get("T", 1)))
        _room(s, [_word_room(case["N"])] * case.get("T", 1))
    elif kind == "batch":
        s["depths"] = [_array(_depth(N, _boxes_of(N), True, seed, 10 + i)) for i, N in enumerate(_sizes(case, case["maps"]))]
        _room(s, [_word_room(N) for N in _sizes(case, case["maps"])])
    elif kind == "frame":
        d = _depth(case["N"], case["boxes"], True, seed, 1)
        s["matrix"], inv = _light(seed)
        p = _to_world(_gbuffer(d, case["W"], case["H"], False, seed, 2), inv)
        s["positions"] = _array(p.reshape(case["H"], case["W"], 4))
        s["vis"] = cp.DeviceArray((case["H"], case["W"]), np.uint8)
        s["image"] = d.cpu().numpy() if case["host"] else _array(d)
        s["container"] = None
    elif kind == "lookup":
        d = _depth(case["N"], case["boxes"], True, seed, 1)
        n = case["count"]
        if case["points"] == "gbuffer":
            W = max(1, int(math.sqrt(n / 2 * 16 / 9)))
            H = -(-n // (2 * W))
            p = _gbuffer(d, W, H, True, seed, 2)[:n]
        else:
            p = _uniform(n, 4, seed, 2)
        s["matrix"] = None
        if case["matrix"]:
            s["matrix"], inv = _light(seed)
            p = _to_world(p, inv)
        s["positions"] = _array(p[:, :case["stride"]])
        s["container"] = _container(d)
        s["vis"] = cp.DeviceArray((n,), np.uint8)
    elif kind == "tiled":
        L = case["L"]
        maps = [_array(_depth(case["N"], case["boxes"], True, seed, 10 + i)) for i in range(L * L)]
        torch.cuda.synchronize()
        keys = [(i, t) for i in range(L * L) for t in range(L)]
        dags, _ = cp.build_batch([maps[i] for i, _ in keys], [(t, L) for _, t in keys])
        c = cp.CompressedShadowContainer(L)
        for (i, t), sh in zip(keys, dags):
            c.set(sh, i % L, i // L, t)
        c.moveToGPU()
        s["container"] = c
        s["positions"] = _array(_uniform(case["count"], 4, seed, 2))
        s["matrix"] = None
        s["vis"] = cp.DeviceArray((case["count"],), np.uint8)
    elif kind == "pcf":
        d = _depth(case["N"], case["boxes"], True, seed, 1)
        s["positions"] = _array(_gbuffer(d, case["W"], case["H"], False, seed, 2))
        s["container"] = _container(d)
        s["container"].setFilterSize(case["f"])
        s["vis"] = cp.DeviceArray((case["W"] * case["H"],), np.float32)
    elif kind == "dagset":
        depths = [_array(_depth(N, _boxes_of(N), True, seed, 10 + i)) for i, N in enumerate(_sizes(case, case["dags"]))]
        torch.cuda.synchronize()
        dags, _ = cp.build_batch(depths)
        for sh in dags:
            sh.setTopLevels(case["top"])
        s["set"] = cp.DagSet(dags)
        s["ndc"] = _array(_uniform(case["count"], 3, seed, 2))
        s["ids"] = None
        if case["ids"]:
            s["ids"] = _array(torch.randint(0, case["dags"], (case["count"],), generator=_rng(seed, 3), device="cuda",
                                            dtype=torch.int32))
        s["vis"] = cp.DeviceArray((case["count"],), np.uint8)
    elif kind == "serve":
        s["server"] = cp.Server(lanes=4, budget_bytes=32 << 30)
        sizes = _sizes(case, case["resident"])
        s["held"] = [_array(_depth(N, _boxes_of(N), True, seed, 10 + i)) for i, N in enumerate(sizes)]
        s["depths"] = [_array(_depth(N, _boxes_of(N), True, seed, 50 + i)) for i, N in enumerate(_sizes(case, case["builds"], 1))]
        counts = _serve_counts(case)
        s["ndc"] = _array(_uniform(sum(counts), 3, seed, 2))
        s["vis"] = cp.DeviceArray((sum(counts),), np.uint8)
        torch.cuda.synchronize()
        tickets = [s["server"].build(d) for d in s["held"]]
        for t in tickets:
            s["server"].wait(t)
        s["plan"], at = [], 0
        for k, n in enumerate(counts):
            s["plan"].append((tickets[k % len(tickets)], n, at))
            at += n
        s["built"] = []
        _room(s, [_word_room(N) for N in _sizes(case, case["builds"], 1)])
    torch.cuda.synchronize()
    return s


def _serve_counts(case):
    r = random.Random(case["mix"] * 17 + 2)
    return [int(2 ** r.uniform(10, 20)) for _ in range(case["lookups"])]


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "build":
        mm = cp.MinMaxHierarchy(s["depth"], borrow=True)
        sh = cp.CompressedShadow.create(mm)
        mm.close()
        return _keep(s, [sh.handle], s["rooms"])
    if kind == "tile":
        mm = cp.MinMaxHierarchy(s["depth"], borrow=True)
        dags = [cp.CompressedShadow.create(mm, t, case["T"]) for t in range(case["T"])]
        mm.close()
        return _keep(s, [sh.handle for sh in dags], s["rooms"])
    if kind == "batch":
        dags, _ = cp.build_batch(s["depths"])
        return _keep(s, [sh.handle for sh in dags], s["rooms"])
    if kind == "frame":
        mm = cp.MinMaxHierarchy(s["image"]) if case["host"] else cp.MinMaxHierarchy(s["image"], borrow=True)
        c = cp.CompressedShadowContainer(cp.CompressedShadow.create(mm))
        mm.close()
        c.moveToGPU()
        old, s["container"] = s["container"], c
        if old is not None:
            old.close()
        return _tensor(c.evaluate_image(s["positions"], s["matrix"], s["vis"]))
    if kind in ("lookup", "tiled"):
        return _tensor(s["container"].evaluate(s["positions"], s["matrix"], s["vis"]))
    if kind == "pcf":
        return _tensor(s["container"].evaluate_pcf(s["positions"], None, s["vis"]))
    if kind == "dagset":
        return _tensor(s["set"].evaluate(s["ndc"], s["ids"], s["vis"]))
    srv = s["server"]
    srv.ctx.synchronize()  # the words of the last burst's DAGs were copied
    for t in s["built"]:
        srv.release(t)
    builds = [srv.build(d) for d in s["depths"]]
    lookups = [srv.lookup(dag, s["ndc"], s["vis"], n, at, at) for dag, n, at in s["plan"]]
    for t in lookups + builds:
        srv.wait(t)
    s["built"], handles = builds, []
    for t in builds:
        handles.append(ctypes.c_void_p())
        _lib.call("cpvs_server_dag", srv.handle, t, ctypes.byref(handles[-1]))
    return [_tensor(s["vis"])] + _keep(s, handles, s["rooms"])


def work(case):
    """Depth read once and results written once; DAG words (written by a build, read in part by the
    lookups) depend on the map and are left out, and the arithmetic is integer or negligible."""
    kind = case["kind"]
    if kind in ("build", "tile"):
        b = 4 * case["N"] ** 2
    elif kind == "batch":
        b = sum(4 * N * N for N in _sizes(case, case["maps"]))
    elif kind == "frame":
        b = 4 * case["N"] ** 2 + 17 * case["W"] * case["H"]
    elif kind == "lookup":
        b = (4 * case["stride"] + 1) * case["count"]
    elif kind == "tiled":
        b = 17 * case["count"]
    elif kind == "pcf":
        b = 20 * case["W"] * case["H"]
    elif kind == "dagset":
        b = (17 if case["ids"] else 13) * case["count"]
    else:
        b = sum(4 * N * N for N in _sizes(case, case["builds"], 1)) + 13 * sum(_serve_counts(case))
    return {"bytes": float(b), "flops": 0.0}


def _path(v, R):
    """traverse.cs's quantisation of one NDC coordinate, in its float32 steps."""
    return (((v + 1.0) * 0.5) * float(R - 1)).clamp_(0.0, float(R - 1)).to(torch.int64)


def exact(case, seed):
    """The filtered visibilities by definition: the share of the f x f cells around each point's
    path that lie in front of the map's depth.  Every other output is whole numbers."""
    if case["kind"] != "pcf":
        return None
    N, f = case["N"], case["f"]
    d = _depth(N, case["boxes"], True, seed, 1)
    p = _gbuffer(d, case["W"], case["H"], False, seed, 2)
    x, y, z = (_path(p[:, k].clone(), N) for k in range(3))
    deep = d.double() * N
    lit = torch.zeros(p.shape[0], dtype=torch.float64, device="cuda")
    lo = -((f - 1) // 2)
    for a in range(f):
        for b in range(f):
            ty, tx = (y + lo + a).clamp_(0, N - 1), (x + lo + b).clamp_(0, N - 1)
            lit += (z.double() + 0.5 <= deep[ty, tx]).double()
    return lit / (f * f)
