#!/usr/bin/env python3
"""Headline benchmark: precomputed-voxelized-shadow build + lookup on one MI355X.

Workload (default): an 8192 x 8192 float32 light-space depth map (tilted plane + 512 boxes +
4-octave value noise, the 8192^3-voxel configuration) and 16,588,800 light-space queries of a
synthetic 3840 x 2160 G-buffer (per pixel one point on the surface, one jittered +-2 voxels).
Depth map and queries are generated on the device and are resident in HBM before timing.

One step = MinMaxHierarchy + CompressedShadow::create of the map (depth in HBM -> DAG words in
HBM), CompressedShadowContainer copyToGPU, and one evaluate() of all queries.

Prints one JSON line.  value = build throughput in Mtexels/s (N^2 depth texels per build);
the lookup rate, p50/p99 latencies, the dominant kernel's roofline and the CPU baseline (the
oracle timed on this machine's host cores) ride along in the same line.
"""
import argparse
import ctypes
import json
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "DAG build Mvoxel-texels/s + G lookups/s; p50/p99 latency, batched vs plain"
HBM_PEAK_GBS = 8000.0
SEED0 = 0x43505653


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def pct(xs, p):
    xs = sorted(xs)
    if not xs:
        return None
    k = (len(xs) - 1) * p / 100.0
    lo, hi = int(k), min(int(k) + 1, len(xs) - 1)
    return xs[lo] + (xs[hi] - xs[lo]) * (k - lo)


def table_slots(n):
    """Slots of a merge table for n keys (build_parts.hpp's table_slots)."""
    return max(1024, n + n // 2 + 1)


def leaf_waves_bytes(N, nodes_leaf):
    """Algorithmic bytes of the leaf kernels: the 8x8 depth block of every level-3 column (256 B) and,
    per leaf node, its breadth-first index read and its run head's index written (8 B).  The first
    node of each run also writes its mask and leafmasks; those bytes are left out, so the figure is
    a lower bound.  The kernels also clear the merge tables (cleared_table_bytes), which is not part of
    the leaf computation."""
    return 256 * (N // 8) ** 2 + 8 * nodes_leaf


def cleared_table_bytes(nodes):
    """The merge tables cleared at the end of the first leaf kernel (8 B per slot): those of the levels
    below the first with more than 4096 nodes from the root down, by build_parts.hpp's size rules (a
    quarter of the leaves and half of the inner nodes from 2^20 on, inner tables below 2^17 nodes at most
    a quarter full).  nodes: per octree level, leaves at level 2."""
    levels = [int(c) for c in nodes]
    top = max(L for L, c in enumerate(levels) if c)
    while top >= 3 and levels[top] <= 4096:
        top -= 1
    slots = 0
    for L in range(2, top + 1):
        c = levels[L]
        if L == 2:
            slots += table_slots(c // 4 if c >= 1 << 20 else c)
        else:
            slots += table_slots(c * 8 // 3 if c < 1 << 17 else c // 2 if c >= 1 << 20 else c)
    return 8 * slots


def host_cpu():
    """The host's CPU: logical CPUs, those this process may run on, and the model name."""
    model = None
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    aff = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    return {"nproc": os.cpu_count(), "usable_cpus": aff, "model": model}


FAITHFUL_CHILD = r"""
import sys, time
sys.path.insert(0, {root!r})
import oracle as O
D = O.gen_depth({N}, {seed}, {boxes}, {noise})
p = O.Pyramid(D)
print("start", flush=True)
t0 = time.perf_counter()
w, n = O.create(p, 0, 1, merge_mode=0)
print("done", time.perf_counter() - t0, len(w), flush=True)
"""


def time_faithful_create(N, seed, boxes, noise, cap_s):
    """The reference's own create(): its linear-search mergeLevel (O(n*u),
    src/CompressedShadowUtil.h:154-182), in the oracle, in a child process stopped after cap_s
    seconds of create().  Returns (seconds or None when capped, words or None)."""
    import subprocess
    code = FAITHFUL_CHILD.format(root=ROOT, N=N, seed=seed, boxes=boxes, noise=noise)
    proc = subprocess.Popen([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True)
    try:
        first = proc.stdout.readline()  # map generated, pyramid built: create() starts now
        if not first.startswith("start"):
            proc.kill()
            proc.wait()
            return None, None
        out, _ = proc.communicate(timeout=cap_s)
        parts = out.split()
        return float(parts[1]), int(parts[2])
    except subprocess.TimeoutExpired:
        proc.kill()
        proc.wait()
        return None, None


def pyramid_root_bytes(N):
    """k_pyr_tile root launch: read the N^2 depth map, write pyramid levels 3..6 as (min,max)."""
    return 4 * N * N + 8 * sum((N >> L) ** 2 for L in range(3, 7))


def load_traffic(N):
    """HBM bytes per launch measured by rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE on this workload
    (committed summary, calibrated against a device copy of known size); {} if not measured."""
    path = os.path.join(ROOT, "profiles", f"c1_{N}_traffic.txt")
    out = {}
    if os.path.exists(path):
        for line in open(path):
            if line.startswith("#") or not line.strip():
                continue
            name, fb, wb = line.rsplit(None, 2)  # kernel names may contain spaces
            out[name.strip()] = int(fb) + int(wb)
    return out


def run_tiled(cp, np, ctx, full=65536, tile=8192, boxes=16384, nq=1 << 26, batch_lanes=8):
    """The tiled configuration: full^2 depth as (full/tile)^2 xy tiles, each built into full/tile
    z-tile DAGs (DeferredRenderer.cpp:150-187), one container with the top-level grid, and nq
    uniform lookups.  All 16 GiB of depth are generated on the device before timing."""
    L = full // tile
    stream = ctx.stream
    log(f"[bench] tiled: generating {L * L} tiles of {tile}^2")
    tiles = {}
    for ty in range(L):
        for tx in range(L):
            tiles[(tx, ty)] = cp.gen_depth(full, SEED0 + 2, boxes, True, tx * tile, ty * tile, tile)
    q = cp.gen_queries_uniform(SEED0 + 3, nq, 4)
    vis = cp.DeviceArray((nq,), np.uint8, ctx)
    c = cp.CompressedShadowContainer(L)
    per_dag, sample, sample_s = [], {}, 0.0
    t0 = time.perf_counter()
    for ty in range(L):
        for tx in range(L):
            e0 = ctx.event(stream)
            mm = cp.MinMaxHierarchy(tiles[(tx, ty)], borrow=True)
            e1 = ctx.event(stream)
            pyr_ms = ctx.elapsed_ms(e0, e1)
            for tz in range(L):
                a = ctx.event(stream)
                sh = cp.CompressedShadow.create(mm, tz, L)
                b = ctx.event(stream)
                if len(per_dag) % 37 == 0:  # checked against the batched build below (time not counted)
                    ts = time.perf_counter()
                    sample[(tx, ty, tz)] = sh.getDAG()
                    sample_s += time.perf_counter() - ts
                c.set(sh, tx, ty, tz)
                per_dag.append(ctx.elapsed_ms(a, b) + pyr_ms / L)
                ctx.destroy_event(a)
                ctx.destroy_event(b)
            ctx.destroy_event(e0)
            ctx.destroy_event(e1)
            mm.close()
    ctx.synchronize()
    build_s = time.perf_counter() - t0 - sample_s
    # The same 512 DAGs as one batch (a tile's z-tiles share its pyramid), in the configuration the
    # autotuner picks among forests and one-map-per-chain lanes.  The words of every 37th plain DAG
    # are compared with the batched one's.
    keys = [(tx, ty, tz) for ty in range(L) for tx in range(L) for tz in range(L)]
    bd, bt = [tiles[(tx, ty)] for tx, ty, _ in keys], [(tz, L) for _, _, tz in keys]
    cands = [cp.batch_config(lanes=batch_lanes, forest_mtexels=0)] + \
        [cp.batch_config(lanes=ln, forest_mtexels=mt) for ln in (1, 2, 4) for mt in (64, 256, 512, 1024)] + \
        [cp.batch_config(lanes=ln, forest_mtexels=mt) for ln in (6, 8) for mt in (128, 256, 512)] + \
        [cp.batch_config(lanes=2, forest_mtexels=64, graph=True), cp.batch_config(lanes=3, forest_mtexels=256)]
    best, tune_ms = cp.tune_batch_config(bd, cands, bt)
    cfg = cands[best]
    log(f"[bench] tiled: tuner picked {cfg.as_dict()} ({[round(m, 1) for m in tune_ms]} ms)")
    runs = []
    for _ in range(3):
        t0 = time.perf_counter()
        batch, _ = cp.build_batch(bd, bt, config=cfg)
        ctx.synchronize()
        runs.append(time.perf_counter() - t0)
        if len(runs) < 3:
            for sh in batch:
                sh.close()
    batch_s = sorted(runs)[1]
    same = all(np.array_equal(batch[keys.index(k)].getDAG(), w) for k, w in sample.items())
    for sh in batch:
        sh.close()
    for d in tiles.values():
        d.free()
    # the lookup top table tuned on the queries (untimed), then the host side freed (moveToGPU)
    top_set, top_ms = c.tuneTopLevels(q, candidates=(-1, 0, 3, 4, 5), visibilities=vis)
    c.freeOnCPU()
    dl, gl, words = c.info()
    top_levels = c.top_levels()
    c.evaluate(q, None, vis)
    ctx.synchronize()
    lk = []
    for _ in range(3):
        a = ctx.event(stream)
        c.evaluate(q, None, vis)
        b = ctx.event(stream)
        lk.append(ctx.elapsed_ms(a, b))
        ctx.destroy_event(a)
        ctx.destroy_event(b)
    c.close()
    q.free()
    vis.free()
    return {"workload": f"{full}x{full} depth ({L}x{L} tiles of {tile}^2, {boxes} boxes + noise), "
                        f"{L}^3 = {L ** 3} z-tile DAGs, {nq} uniform lookups",
            "dags": L ** 3, "dag_words": words, "grid_levels": gl,
            "build_s": round(build_s, 4), "Mtexels_per_s": round(full * full / build_s / 1e6, 1),
            "batched_build_s": round(batch_s, 4), "batched_Mtexels_per_s": round(full * full / batch_s / 1e6, 1),
            "batch_config": cfg.as_dict(),
            "tune_ms": {json.dumps(c.as_dict(), sort_keys=True): round(m, 2) for c, m in zip(cands, tune_ms)},
            "batched_words_identical": bool(same),
            "dag_build_ms_p50": round(pct(per_dag, 50), 3), "dag_build_ms_p99": round(pct(per_dag, 99), 3),
            "lookup_G_per_s": round(nq / (min(lk) * 1e-3) / 1e9, 3),
            "lookup_top_table": {"setting": top_set, "levels": top_levels,
                                 "tune_ms": {str(k): round(v, 4) for k, v in top_ms.items()}}}


def run_c0(cp, np, ctx, N=1024, boxes=32, nq=1 << 20, reps=20):
    """The 1024^2 configuration: plane + 32 boxes (no noise), 1,048,576 uniform lookups."""
    stream = ctx.stream
    d = cp.gen_depth(N, SEED0, boxes, False)
    q = cp.gen_queries_uniform(SEED0, nq, 4)
    vis = cp.DeviceArray((nq,), np.uint8, ctx)
    mm = cp.MinMaxHierarchy(d, borrow=True)
    c = cp.CompressedShadowContainer(cp.CompressedShadow.create(mm))
    top_set, top_ms = c.tuneTopLevels(q, candidates=(-1, 0, 4, 5, 6, 7, 8), visibilities=vis)  # untimed
    c.close()
    mm.close()
    bms, lms = [], []
    for it in range(reps + 3):
        e0 = ctx.event(stream)
        mm = cp.MinMaxHierarchy(d, borrow=True)
        cs = cp.CompressedShadow.create(mm)
        e1 = ctx.event(stream)
        words = cs.num_words()
        c = cp.CompressedShadowContainer(cs)
        c.setTopLevels(top_set)
        c.copyToGPU()
        e2 = ctx.event(stream)
        c.evaluate(q, None, vis)
        e3 = ctx.event(stream)
        if it >= 3:
            bms.append(ctx.elapsed_ms(e0, e1))
            lms.append(ctx.elapsed_ms(e2, e3))
        for e in (e0, e1, e2, e3):
            ctx.destroy_event(e)
        c.close()
        mm.close()
    d.free()
    q.free()
    vis.free()
    return {"workload": f"{N}x{N} depth (plane + {boxes} boxes), {nq} uniform lookups",
            "build_ms_p50": round(pct(bms, 50), 4), "build_ms_p99": round(pct(bms, 99), 4),
            "Mtexels_per_s": round(N * N / (pct(bms, 50) * 1e-3) / 1e6, 1), "dag_words": words,
            "lookup_G_per_s": round(nq / (pct(lms, 50) * 1e-3) / 1e9, 3),
            "lookup_top_table": {"setting": top_set, "tune_ms": {str(k): round(v, 4) for k, v in top_ms.items()}}}


def splitmix64(seed):
    """splitmix64 stream (the generator's PRNG): yields 64-bit ints."""
    x = seed & 0xFFFFFFFFFFFFFFFF
    M = 0xFFFFFFFFFFFFFFFF
    while True:
        x = (x + 0x9E3779B97F4A7C15) & M
        z = x
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M
        yield z ^ (z >> 31)


def run_batched(cp, np, ctx, maps=256, kmin=8, kmax=13, qper=1 << 20, reps=3):
    """Many maps: `maps` depth maps of side 2^k, k uniform in [kmin, kmax] (boxes 32*(N/1024)^2,
    at least 1, plus noise; map i seeded SEED0 + 3 + 1000*(i+1)), built plainly (one
    MinMaxHierarchy + create chain after another on one stream, as the reference's loop) and as one
    batch (cpvs_build_batch, lane count chosen by cpvs_tune_batch).  Then maps*qper uniform
    lookups: plainly one launch per DAG over its own qper queries, and batched as one launch
    over all of them interleaved round-robin (query j -> DAG j mod maps) through a DAG set.
    Plain lookups read each DAG's queries from the interleaved buffer (stride maps*3 floats); the
    same on a map-major copy made before timing is reported beside them.  Every map arrives at
    t=0; its latency is its completion time."""
    seed = SEED0 + 3
    rng = splitmix64(seed)
    sizes = [1 << (kmin + next(rng) % (kmax - kmin + 1)) for _ in range(maps)]
    log(f"[bench] batched: generating {maps} maps (sizes {sorted(set(sizes))})")
    depths = []
    for i, N in enumerate(sizes):
        depths.append(cp.gen_depth(N, seed + 1000 * (i + 1), max(1, (32 * N * N) // (1024 * 1024)), True))
    ctx.synchronize()
    texels = float(sum(N * N for N in sizes))

    def plain_once():
        out, done = [], []
        t0 = time.perf_counter()
        for d in depths:
            mm = cp.MinMaxHierarchy(d, borrow=True)
            out.append(cp.CompressedShadow.create(mm))
            mm.close()
            done.append((time.perf_counter() - t0) * 1e3)
        ctx.synchronize()
        return out, done, time.perf_counter() - t0

    def batch_once():
        t0 = time.perf_counter()
        out, done = cp.build_batch(depths)
        return out, list(done), time.perf_counter() - t0

    # warm-up of the plain path (arena sizing), then the autotuner picks the batch configuration:
    # forests (many maps through one launch chain) of several sizes on 1-4 lanes, hipGraph capture,
    # and one map per launch chain on 4 or 8 lanes.
    for sh in plain_once()[0]:
        sh.close()
    cands = [cp.batch_config(lanes=ln, forest_mtexels=0) for ln in (4, 8)] + \
        [cp.batch_config(lanes=ln, forest_mtexels=mt) for ln in (1, 2, 4) for mt in (64, 256, 1024)] + \
        [cp.batch_config(lanes=2, forest_mtexels=256, graph=True)]
    bi, tms = cp.tune_batch_config(depths, cands)
    best = cands[bi].as_dict()
    tune_ms = {json.dumps(c.as_dict(), sort_keys=True): m for c, m in zip(cands, tms)}
    lane_ms = min(m for c, m in zip(cands, tms) if c.forest_mtexels == 0)
    log(f"[bench] batched: tuner picked {best} ({[round(m, 1) for m in tms]} ms)")
    plain_runs, batch_runs = [], []
    plain, batch = None, None
    for r in range(reps):
        sh, done, sec = plain_once()
        plain_runs.append((sec, done))
        if r < reps - 1:
            for x in sh:
                x.close()
        else:
            plain = sh
        sh, done, sec = batch_once()
        batch_runs.append((sec, done))
        if r < reps - 1:
            for x in sh:
                x.close()
        else:
            batch = sh
        log(f"[bench] batched: rep {r}: plain {plain_runs[-1][0] * 1e3:.1f} ms, batch {sec * 1e3:.1f} ms")
    p_sec, p_done = sorted(plain_runs)[len(plain_runs) // 2]
    b_sec, b_done = sorted(batch_runs)[len(batch_runs) // 2]
    words_plain = [x.num_words() for x in plain]
    words_batch = [x.num_words() for x in batch]
    same = words_plain == words_batch
    small = sorted(range(maps), key=lambda i: sizes[i])[:32]
    for i in small:
        same = same and bool(np.array_equal(plain[i].getDAG(), batch[i].getDAG()))
    for x in plain:
        x.close()
    for d in depths:
        d.free()

    # lookups: the same maps*qper points, interleaved round-robin (query j -> DAG j mod maps)
    nq = maps * qper
    stream = ctx.stream
    q_rr = cp.gen_queries_uniform(seed + 17, nq, 3)
    vis_rr = cp.DeviceArray((nq,), np.uint8, ctx)
    vis_st = cp.DeviceArray((nq,), np.uint8, ctx)
    q_mm = cp.DeviceArray((nq, 3), np.float32, ctx)
    for i in range(maps):  # map-major copy of the same points: block i = points i, i+maps, ...
        cp._lib.call("cpvs_gen_queries_uniform_range", ctx.handle, ctypes.c_void_p(q_mm.ptr.value + 12 * qper * i),
                     seed + 17, i, maps, qper, 3, None)
    vis_mm = cp.DeviceArray((nq,), np.uint8, ctx)
    # Each DAG's lookup top table, one setting for all, picked by timing the batched lookups
    # (untimed); the plain and the batched lookups below both read the tables.
    top_ms = {}
    for k in (0, 2, 3, 4, 5):
        for sh in batch:
            sh.setTopLevels(k)
        ds = cp.DagSet(batch)
        ds.evaluate(q_rr, None, vis_rr, stream)
        e0 = ctx.event(stream)
        ds.evaluate(q_rr, None, vis_rr, stream)
        e1 = ctx.event(stream)
        top_ms[k] = ctx.elapsed_ms(e0, e1)
        for e in (e0, e1):
            ctx.destroy_event(e)
        ds.close()
    top_set = min(top_ms, key=top_ms.get)
    for sh in batch:
        sh.setTopLevels(top_set)
    log(f"[bench] batched: DAG top tables {top_set} levels ({ {k: round(v, 2) for k, v in top_ms.items()} } ms)")
    dset = cp.DagSet(batch)
    lk = {"plain": [], "plain_grouped": [], "batched": []}

    def plain_pass(q, qstride, qstep, out):
        for i, sh in enumerate(batch):
            cp._lib.call("cpvs_dag_evaluate", sh.handle, ctypes.c_void_p(q.ptr.value + qstep * i), qstride, qper,
                         ctypes.c_void_p(out.ptr.value + qper * i), stream)

    for r in range(reps + 1):
        ev = [ctx.event(stream)]
        plain_pass(q_rr, 3 * maps, 12, vis_st)  # one launch per DAG over its strided queries
        ev.append(ctx.event(stream))
        plain_pass(q_mm, 3, 12 * qper, vis_mm)  # the same on a pre-grouped copy
        ev.append(ctx.event(stream))
        dset.evaluate(q_rr, None, vis_rr, stream)  # one launch over all, DAG set round-robin
        ev.append(ctx.event(stream))
        if r:
            lk["plain"].append(ctx.elapsed_ms(ev[0], ev[1]))
            lk["plain_grouped"].append(ctx.elapsed_ms(ev[1], ev[2]))
            lk["batched"].append(ctx.elapsed_ms(ev[2], ev[3]))
        for e in ev:
            ctx.destroy_event(e)
    vr = vis_rr.numpy().reshape(qper, maps).T
    same_lookup = bool(np.array_equal(vr, vis_mm.numpy().reshape(maps, qper))) and \
        bool(np.array_equal(vr, vis_st.numpy().reshape(maps, qper)))
    dset.close()
    for x in batch:
        x.close()
    for a in (q_rr, vis_rr, vis_st, q_mm, vis_mm):
        a.free()
    rate = {k: nq / (min(v) * 1e-3) / 1e9 for k, v in lk.items()}
    return {"workload": f"{maps} maps of 2^k x 2^k, k uniform in [{kmin},{kmax}] (boxes 32*(N/1024)^2 + noise), "
                        f"{nq} uniform lookups ({qper} per map, interleaved round-robin)",
            "maps": maps, "texels": int(texels), "config": best,
            "tune_ms": {k: round(v, 2) for k, v in tune_ms.items()},
            "lane_mode_best_ms": round(lane_ms, 2),
            "plain_build_ms": round(p_sec * 1e3, 2), "batched_build_ms": round(b_sec * 1e3, 2),
            "plain_Mtexels_per_s": round(texels / p_sec / 1e6, 1),
            "batched_Mtexels_per_s": round(texels / b_sec / 1e6, 1),
            "build_speedup": round(p_sec / b_sec, 2),
            "plain_latency_ms_p50": round(pct(p_done, 50), 2), "plain_latency_ms_p99": round(pct(p_done, 99), 2),
            "batched_latency_ms_p50": round(pct(b_done, 50), 2), "batched_latency_ms_p99": round(pct(b_done, 99), 2),
            "dag_words": int(sum(words_batch)), "words_identical": bool(same),
            "lookup_plain_G_per_s": round(rate["plain"], 3),
            "lookup_plain_pregrouped_G_per_s": round(rate["plain_grouped"], 3),
            "lookup_batched_G_per_s": round(rate["batched"], 3),
            "lookup_speedup": round(rate["batched"] / rate["plain"], 3),
            "lookup_top_levels": top_set, "lookup_top_tune_ms": {str(k): round(v, 3) for k, v in top_ms.items()},
            "lookups_identical": same_lookup}


def run_serving(cp, np, ctx, nreq=10000, p_build=0.3, kmin=9, kmax=14, warm_per_size=4, load=0.7,
                budget=200 << 30, lanes=4, pressure_budget=32 << 30):
    """Serving: a trace of nreq requests, each a build (probability p_build) of a 2^k map, k uniform
    in [kmin, kmax], or a lookup of 2^U(10,22) uniform points against one of a warm set of
    resident DAGs (warm_per_size per size, built before timing).  Depth maps (one per size) and
    points are generated on the device first.  The trace is served by the serial server (one
    request at a time, the plain path) and by the concurrent server (build lanes + continuous
    lookup batching), first all at once (throughput), then with Poisson arrivals at `load` times
    the serial throughput (latency = submission to completion, per request kind)."""
    import random
    seed = SEED0 + 4
    rng = random.Random(seed)
    sizes = list(range(kmin, kmax + 1))
    log(f"[bench] serving: generating maps 2^{kmin}..2^{kmax} and points")
    depth = {k: cp.gen_depth(1 << k, seed + 1000 * k, max(1, (32 << (2 * k)) >> 20), True) for k in sizes}
    qmax = 1 << 22
    q = cp.gen_queries_uniform(seed + 17, qmax, 3)
    trace = []  # (kind, k or warm index, count, point offset)
    for _ in range(nreq):
        if rng.random() < p_build:
            trace.append((0, rng.choice(sizes), 0, 0))
        else:
            n = int(2 ** rng.uniform(10, 22))
            trace.append((1, rng.randrange(warm_per_size * len(sizes)), n, rng.randrange(0, qmax - n + 1)))
    out_bytes = sum(t[2] for t in trace)
    vis = cp.DeviceArray((out_bytes,), np.uint8, ctx)
    ctx.synchronize()

    def serve(serial, arrivals, budget=budget, kcap=kmax):
        # kcap: builds of larger maps build a 2^kcap map instead, and only sizes up to it are warm.
        srv = cp.Server(lanes=lanes, budget_bytes=budget, serial=serial, ctx=ctx)
        try:
            warm = []
            for k in sizes:
                if k > kcap:
                    continue
                for _ in range(warm_per_size):
                    warm.append(srv.build(depth[k]))
            for t in warm:
                srv.wait(t)
            tickets, kinds, lag = [], [], []
            off = 0
            missed = 0
            t0 = time.perf_counter()
            for (kind, a, n, qo), at in zip(trace, arrivals):
                if at is not None:
                    while True:
                        dt = at - (time.perf_counter() - t0)
                        if dt <= 0:
                            break
                        if dt > 2e-4:
                            time.sleep(dt - 1e-4)
                    lag.append((time.perf_counter() - t0) - at)
                if kind == 0:
                    tickets.append(srv.build(depth[min(a, kcap)]))
                else:
                    try:
                        tickets.append(srv.lookup(warm[a % len(warm)], q, vis, count=n, offset=qo, vis_offset=off))
                    except cp.CpvsError:  # its DAG was evicted under a tight budget: not served
                        missed += 1
                        continue
                    off += n
                kinds.append(kind)
            lat, failed = [], 0
            for t in tickets:
                try:
                    lat.append(srv.wait(t))
                except cp.CpvsError:  # a build the budget could not admit
                    lat.append(None)
                    failed += 1
            lat_kinds = [(x, k) for x, k in zip(lat, kinds) if x is not None]
            sec = time.perf_counter() - t0
            st = srv.stats()
        finally:
            srv.close()
        b = [x for x, k in lat_kinds if k == 0]
        l = [x for x, k in lat_kinds if k == 1]
        return {"s": sec, "req_per_s": len(trace) / sec,
                "build_ms_p50": pct(b, 50), "build_ms_p99": pct(b, 99),
                "lookup_ms_p50": pct(l, 50), "lookup_ms_p99": pct(l, 99),
                "lookup_batches": st["batches"], "lookups": st["lookups"], "evicted": st["evicted"],
                "trims": st["trims"], "lookups_on_evicted": missed, "builds": st["builds"], "failed": failed,
                "submit_lag_ms_p99": pct(lag, 99) * 1e3 if lag else None}

    none = [None] * len(trace)
    thr = {m: serve(m == "serial", none) for m in ("serial", "served")}
    log(f"[bench] serving throughput: {thr}")
    rate = load * thr["serial"]["req_per_s"]
    arr, t = [], 0.0
    for _ in trace:
        t += rng.expovariate(rate)
        arr.append(t)
    lat = {m: serve(m == "serial", arr) for m in ("serial", "served")}
    log(f"[bench] serving latency at {rate:.0f} req/s: {lat}")
    # The same Poisson trace under a budget that forces evictions, with maps of at most 8192^2 (a
    # 16384^2 map of this generator has about 200 M leaf nodes and alone needs some 35 GB of scratch
    # and DAG reservation): the resident DAGs of the builds outgrow the budget, so least recently
    # used DAGs are evicted (no device synchronisation on that path).
    press = {m: serve(m == "serial", arr, pressure_budget, kcap=min(kmax, 13)) for m in ("serial", "served")}
    log(f"[bench] serving under a {pressure_budget >> 30} GiB budget: {press}")
    vis.free()
    q.free()
    for d in depth.values():
        d.free()

    def r(v):
        return None if v is None else round(v, 3)
    return {"workload": f"{nreq} requests: {p_build:.0%} builds of 2^k maps (k uniform in [{kmin},{kmax}], "
                        f"boxes + noise), lookups of 2^U(10,22) uniform points on one of "
                        f"{warm_per_size * len(sizes)} resident DAGs; HBM budget {budget >> 30} GiB",
            "lanes": lanes,
            "throughput_req_per_s": {m: round(v["req_per_s"], 1) for m, v in thr.items()},
            "throughput_speedup": round(thr["served"]["req_per_s"] / thr["serial"]["req_per_s"], 2),
            "poisson_rate_req_per_s": round(rate, 1),
            "latency_ms": {m: {k: r(v[k]) for k in ("build_ms_p50", "build_ms_p99", "lookup_ms_p50", "lookup_ms_p99")}
                           for m, v in lat.items()},
            "lookup_launches": {m: v["lookup_batches"] for m, v in lat.items()},
            "evicted": {m: v["evicted"] for m, v in lat.items()},
            "submit_lag_ms_p99": {m: r(v["submit_lag_ms_p99"]) for m, v in lat.items()},
            "pressure": {"budget_GiB": pressure_budget >> 30, "max_map": f"{1 << min(kmax, 13)}^2",
                         "latency_ms": {m: {k: r(v[k]) for k in ("build_ms_p50", "build_ms_p99", "lookup_ms_p50",
                                                                  "lookup_ms_p99")} for m, v in press.items()},
                         "req_per_s": {m: round(v["req_per_s"], 1) for m, v in press.items()},
                         "evicted": {m: v["evicted"] for m, v in press.items()},
                         "cache_trims": {m: v["trims"] for m, v in press.items()},
                         "lookups_on_evicted_dags": {m: v["lookups_on_evicted"] for m, v in press.items()},
                         "requests_failed": {m: v["failed"] for m, v in press.items()}}}


def run_tiled_batch_only(cp, ctx, full=65536, tile=8192, boxes=16384, lanes=6, forest_mtexels=128, reps=2):
    """For a kernel trace: the tiled configuration's 512 z-tile DAGs built as one batch `reps`
    times (forests, the given lanes and forest size), after the tiles are generated.  Prints the
    host time of each build."""
    L = full // tile
    tiles = {(tx, ty): cp.gen_depth(full, SEED0 + 2, boxes, True, tx * tile, ty * tile, tile)
             for ty in range(L) for tx in range(L)}
    keys = [(tx, ty, tz) for ty in range(L) for tx in range(L) for tz in range(L)]
    bd, bt = [tiles[(tx, ty)] for tx, ty, _ in keys], [(tz, L) for _, _, tz in keys]
    cfg = cp.batch_config(lanes=lanes, forest_mtexels=forest_mtexels)
    ctx.synchronize()
    out = []
    for _ in range(reps):
        t0 = time.perf_counter()
        batch, _ = cp.build_batch(bd, bt, config=cfg)
        ctx.synchronize()
        out.append(round((time.perf_counter() - t0) * 1e3, 2))
        for sh in batch:
            sh.close()
    for d in tiles.values():
        d.free()
    return {"tiled_batch_ms": out, "config": cfg.as_dict()}


def run_busy_phases(cp, np, ctx, maps=256, kmin=8, kmax=13, config=None):
    """For a kernel trace (rocprofv3 --kernel-trace): the batched configuration's 256 maps built
    plainly (one map after another on one stream), then as one batch (forests), each phase after
    a 0.3 s pause so that --busy-from can tell them apart.  Prints the host times."""
    seed = SEED0 + 3
    rng = splitmix64(seed)
    sizes = [1 << (kmin + next(rng) % (kmax - kmin + 1)) for _ in range(maps)]
    depths = [cp.gen_depth(N, seed + 1000 * (i + 1), max(1, (32 * N * N) // (1024 * 1024)), True)
              for i, N in enumerate(sizes)]
    ctx.synchronize()
    cfg = config or cp.batch_config(lanes=4, forest_mtexels=1024)

    def plain():
        out = []
        for d in depths:
            mm = cp.MinMaxHierarchy(d, borrow=True)
            out.append(cp.CompressedShadow.create(mm))
            mm.close()
        ctx.synchronize()
        return out

    def batch():
        return cp.build_batch(depths, config=cfg)[0]

    for f in (plain, batch):  # warm-up: arenas, lanes
        for sh in f():
            sh.close()
    res = {}
    for name, f in (("plain", plain), ("batched", batch)):
        time.sleep(0.3)
        t0 = time.perf_counter()
        out = f()
        res[name + "_ms"] = round((time.perf_counter() - t0) * 1e3, 2)
        for sh in out:
            sh.close()
    time.sleep(0.3)
    res["config"] = cfg.as_dict()
    return res


def busy_from(db_path, gap_ms=100.0):
    """GPU-busy fraction of each phase of a rocprofv3 kernel trace (its SQLite results): phases are
    separated by idle gaps of at least gap_ms; busy = the union of kernel intervals over the span
    from a phase's first kernel start to its last kernel end."""
    import sqlite3
    con = sqlite3.connect(db_path)
    rows = con.execute("select start, end from kernels order by start").fetchall()
    phases, cur = [], []
    last_end = None
    for st, en in rows:
        if last_end is not None and st - last_end > gap_ms * 1e6:
            phases.append(cur)
            cur = []
        cur.append((st, en))
        last_end = en if last_end is None else max(last_end, en)
    if cur:
        phases.append(cur)
    out = []
    for ph in phases:
        busy, s0, e0 = 0, None, None
        for st, en in ph:  # union of intervals (sorted by start)
            if e0 is None or st > e0:
                if e0 is not None:
                    busy += e0 - s0
                s0, e0 = st, en
            else:
                e0 = max(e0, en)
        busy += e0 - s0
        span = max(en for _, en in ph) - ph[0][0]
        out.append({"kernels": len(ph), "span_ms": round(span / 1e6, 3), "busy_ms": round(busy / 1e6, 3),
                    "busy_fraction": round(busy / span, 3)})
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--N", type=int, default=8192)
    ap.add_argument("--boxes", type=int, default=512)
    ap.add_argument("--top-levels", type=int, default=None,
                    help="lookup top-table setting of the headline container (default: tuned on the queries)")
    ap.add_argument("--width", type=int, default=3840)
    ap.add_argument("--height", type=int, default=2160)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-tiled", action="store_true", help="skip the 65536^2 tiled configuration")
    ap.add_argument("--no-batched", action="store_true", help="skip the 256-map batched configuration")
    ap.add_argument("--no-serving", action="store_true", help="skip the serving configuration")
    ap.add_argument("--no-check", action="store_true", help="skip the brute-force check of the headline lookups")
    ap.add_argument("--no-c0", action="store_true", help="skip the 1024^2 configuration")
    ap.add_argument("--faithful-cap", type=float, default=20.0,
                    help="seconds the faithful (linear-search) create() may run at the headline map")
    ap.add_argument("--busy-phases", action="store_true",
                    help="only build the 256-map batch plainly and batched, paused apart, for a kernel trace")
    ap.add_argument("--tiled-batch-only", action="store_true",
                    help="only build the tiled map's 512 DAGs as one batch twice, for a kernel trace")
    ap.add_argument("--busy-from", metavar="RESULTS_DB",
                    help="print the GPU-busy fraction of each phase of a rocprofv3 kernel trace, and exit")
    args = ap.parse_args()
    if args.busy_from:
        print(json.dumps(busy_from(args.busy_from)))
        return

    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {args.gpus}, WORLD_SIZE={world}): each DAG build "
              f"and lookup batch is independent per GPU, and this build measures the single-GPU path.",
              file=sys.stderr)
        sys.exit(2)

    import numpy as np

    import cpvs_amd as cp

    ctx = cp.default_context()
    if args.busy_phases:
        print(json.dumps(run_busy_phases(cp, np, ctx)), flush=True)
        return
    if args.tiled_batch_only:
        print(json.dumps(run_tiled_batch_only(cp, ctx)), flush=True)
        return
    N = args.N
    log(f"[bench] generating {N}^2 depth map and {2 * args.width * args.height} queries on the device")
    depth = cp.gen_depth(N, SEED0 + 1, args.boxes, True)
    queries = cp.gen_queries_gbuffer(depth, SEED0 + 17, args.width, args.height)
    nq = queries.shape[0]
    vis = cp.DeviceArray((nq,), np.uint8, ctx)
    stream = ctx.stream

    # Device copy of known size: achievable HBM bandwidth, and the reference point for scaling
    # rocprof FETCH_SIZE / WRITE_SIZE counters.
    copy_bytes = 256 << 20
    src = cp.DeviceArray((copy_bytes // 4,), np.float32, ctx)
    dst = cp.DeviceArray((copy_bytes // 4,), np.float32, ctx)
    copy_ms = []
    for _ in range(5):
        c0 = ctx.event(stream)
        cp._lib.call("cpvs_device_copy", ctx.handle, dst.ptr, src.ptr, copy_bytes, stream)
        c1 = ctx.event(stream)
        copy_ms.append(ctx.elapsed_ms(c0, c1))
        ctx.destroy_event(c0)
        ctx.destroy_event(c1)
    copy_gbs = 2 * copy_bytes / (min(copy_ms) * 1e-3) / 1e9
    src.free()
    dst.free()
    log(f"[bench] device copy of {copy_bytes >> 20} MiB: {min(copy_ms):.3f} ms = {copy_gbs:.0f} GB/s (read + write)")

    # The container's lookup top table, tuned on these queries before the steps (untimed): every
    # step's container is built with the setting it picks.
    if args.top_levels is None:
        mm = cp.MinMaxHierarchy(depth, borrow=True)
        c = cp.CompressedShadowContainer(cp.CompressedShadow.create(mm))
        top_set, top_ms = c.tuneTopLevels(queries, candidates=(-1, 0, 4, 5, 6, 7, 8), visibilities=vis)
        c.close()
        mm.close()
        log(f"[bench] top table: tuner picked {top_set} ({ {k: round(v, 4) for k, v in top_ms.items()} } ms)")
    else:
        top_set, top_ms = args.top_levels, {}

    build_ms, lookup_ms, step_ms, container_ms = [], [], [], []
    words = None
    dag_words_host = None
    levels = None
    top_levels = None
    for it in range(args.warmup + args.steps):
        t0 = time.perf_counter()
        e0 = ctx.event(stream)
        mm = cp.MinMaxHierarchy(depth, borrow=True)
        cs = cp.CompressedShadow.create(mm)
        e1 = ctx.event(stream)
        if words is None:
            words = cs.num_words()
            levels = cs.level_stats()
            dag_words_host = cs.getDAG() if not args.no_cpu_baseline else None
        c = cp.CompressedShadowContainer(cs)
        c.setTopLevels(top_set)
        c.copyToGPU()
        e2 = ctx.event(stream)
        c.evaluate(queries, None, vis)
        e3 = ctx.event(stream)
        b = ctx.elapsed_ms(e0, e1)
        lk = ctx.elapsed_ms(e2, e3)
        cm = ctx.elapsed_ms(e1, e2)
        top_levels = c.top_levels()
        t1 = time.perf_counter()
        for e in (e0, e1, e2, e3):
            ctx.destroy_event(e)
        c.close()
        mm.close()
        if it >= args.warmup:
            build_ms.append(b)
            lookup_ms.append(lk)
            container_ms.append(cm)
            step_ms.append((t1 - t0) * 1e3)
        log(f"[bench] step {it}: build {b:.3f} ms, lookup {lk:.3f} ms, step {(t1 - t0) * 1e3:.2f} ms")

    texels = float(N) * N
    build_rate = texels * len(build_ms) / (sum(build_ms) * 1e-3) / 1e6  # Mtexels/s
    lookup_rate = nq * len(lookup_ms) / (sum(lookup_ms) * 1e-3) / 1e9  # G lookups/s

    # The reference's boundary takes a host image (MinMaxHierarchy(const ImageF&)): the same build
    # from the depth map in pageable host memory, PCIe copy included, on the host clock.
    depth_host = depth.numpy()
    host_ms = []
    for _ in range(4):
        ctx.synchronize()
        t0 = time.perf_counter()
        mm = cp.MinMaxHierarchy(depth_host)
        cs = cp.CompressedShadow.create(mm)
        ctx.synchronize()
        host_ms.append((time.perf_counter() - t0) * 1e3)
        cs.close()
        mm.close()
    host_ms = host_ms[1:]  # the first run pays the host pages' first touch
    del depth_host
    host_input = {"build_ms_min": round(min(host_ms), 3), "build_ms_mean": round(statistics.mean(host_ms), 3),
                  "Mtexels_per_s": round(texels / (min(host_ms) * 1e-3) / 1e6, 1),
                  "note": "depth in pageable host memory: H2D copy + pyramid + create, host clock"}
    log(f"[bench] host-input build: {host_input}")

    # Per-kernel timing (HIP events around every launch on the context stream), separate pass.
    ctx.profile(-1)
    ctx.profile(1)
    prof_steps = 3
    for _ in range(prof_steps):
        mm = cp.MinMaxHierarchy(depth, borrow=True)
        cs = cp.CompressedShadow.create(mm)
        c = cp.CompressedShadowContainer(cs)
        c.setTopLevels(top_set)
        c.copyToGPU()
        c.evaluate(queries, None, vis)
        ctx.synchronize()
        c.close()
        mm.close()
    ctx.profile(0)
    prof = ctx.profile_read()
    ctx.profile(-1)
    build_kernels = {k: v for k, v in prof.items() if not k.startswith("evaluate")}
    dominant = max(build_kernels.items(), key=lambda kv: kv[1][0])
    log("[bench] kernel totals over %d profiled steps:" % prof_steps)
    for k, (ms, cnt) in sorted(prof.items(), key=lambda kv: -kv[1][0]):
        log(f"    {k:18s} {ms / prof_steps:9.3f} ms/step  {cnt // prof_steps:5d} launches/step")

    nodes, uniq = levels
    leaf_name = "leaf_lanes" if "leaf_lanes" in prof else "leaf_waves"
    algo = {  # algorithmic bytes per profiled step of the kernels with a closed form
        leaf_name: leaf_waves_bytes(N, int(nodes[2])),
        "pyr_tile_root": pyramid_root_bytes(N),
        "evaluate4": 17 * nq,
    }

    traffic = load_traffic(N)

    # The leaf level takes two launches: smooth columns one per lane, then walls one per wave.
    leaf_parts = [k for k in ("leaf_lanes", "leaf_waves") if k in prof]

    def roof(name):
        ms, cnt = prof[name]
        if name == "leaf_lanes":
            ms = sum(prof[k][0] for k in leaf_parts)
        per_launch_ms = ms / cnt
        bytes_per_launch = algo[name] / (cnt / prof_steps)
        ach = bytes_per_launch / (per_launch_ms * 1e-3) / 1e9
        return {"kernel": name, "bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(ach / HBM_PEAK_GBS, 4), "traffic": (sum(traffic[k] for k in leaf_parts if k in traffic) or None) if name == "leaf_lanes"
                else traffic.get(name),
                "avg_launch_us": round(per_launch_ms * 1e3, 2),
                "bytes_per_launch": int(bytes_per_launch)}

    rname = dominant[0] if dominant[0] in algo else leaf_name
    roofline = roof(rname)
    if rname == leaf_name:
        # The HBM roofline is the ceiling; what holds the kernels below it:
        roofline["limiter"] = ("leaf_lanes: depth loads, then scattered stores of leafmask rows (a fifth of its time); "
                               "leaf_waves: scattered stores of run heads; not HBM bandwidth")
        roofline["table_clear_bytes"] = cleared_table_bytes(nodes)
    pyramid_roofline = roof("pyr_tile_root")
    lookup_roofline = roof("evaluate4")
    # Dependent gathers from a cache-resident DAG: set by load throughput and L2 locality, not HBM.
    lookup_roofline["bound"] = "L2 (dependent gathers; DAG cache-resident)"

    tiled = None
    if not args.no_tiled:
        tiled = run_tiled(cp, np, ctx)
        log(f"[bench] released {ctx.release_scratch() >> 20} MiB of scratch")
        log(f"[bench] tiled: {tiled}")

    batched = None
    if not args.no_batched:
        batched = run_batched(cp, np, ctx)
        log(f"[bench] batched: {batched}")
        log(f"[bench] released {ctx.release_scratch() >> 20} MiB of scratch")

    serving = None
    if not args.no_serving:
        serving = run_serving(cp, np, ctx)
        log(f"[bench] serving: {serving}")

    # Every one of the headline lookups against the brute-force depth compare (outside the timed
    # region): the result of the last timed evaluate().
    check = None
    if not args.no_check:
        import oracle as O
        D = depth.numpy()
        qh = queries.numpy()
        vh = vis.numpy()
        R = np.float32((1 << (len(levels[0]) - 1)) - 1)
        same = True
        for lo in range(0, nq, 1 << 22):
            hi = min(lo + (1 << 22), nq)
            p = (((qh[lo:hi, :3] + np.float32(1)) * np.float32(0.5)) * R).astype(np.int64)
            same = same and bool(np.array_equal(vh[lo:hi], O.brute_visible(D, 1, p[:, 0], p[:, 1], p[:, 2])))
        check = {"lookups_equal_brute_force": same, "queries_checked": nq, "lit_fraction": round(float(vh.mean()), 4)}
        del qh, vh
        log(f"[bench] headline lookups vs brute force: {check}")

    c0 = None
    if not args.no_c0:
        c0 = run_c0(cp, np, ctx)
        log(f"[bench] 1024^2: {c0}")

    cpu = None
    if not args.no_cpu_baseline:
        import oracle as O
        hc = host_cpu()
        log(f"[bench] CPU baseline on {hc}: oracle create() (hash merge, identical words) on the same map")
        D = depth.numpy()
        t0 = time.perf_counter()
        pyr = O.Pyramid(D)
        w, _ = O.create(pyr, 0, 1, merge_mode=1)
        t1 = time.perf_counter()
        words_equal = None
        if dag_words_host is not None:
            words_equal = bool(np.array_equal(w, dag_words_host))
        assert len(w) == words, (len(w), words)
        threads = max(1, min(16, hc["usable_cpus"]))  # the box's CPU share for one GPU is 16
        sample = nq
        qh = queries.numpy()
        grid = O.top_level_grid([w])
        t2 = time.perf_counter()
        O.evaluate(w, grid, len(nodes), 0, qh, nthreads=threads)
        t3 = time.perf_counter()
        t4 = time.perf_counter()
        O.evaluate(w, grid, len(nodes), 0, qh[:2_000_000], nthreads=1)
        t5 = time.perf_counter()
        del qh
        # The reference's create() with its own linear-search merge: timed at 1024^2 (plane + 32
        # boxes), and stopped after a cap at the headline map, where it needs hours.
        log("[bench] CPU baseline: faithful create() (linear-search mergeLevel) at 1024^2 and, capped, at the headline map")
        f0_s, f0_words = time_faithful_create(1024, SEED0, 32, False, 300)
        f1_s, _ = time_faithful_create(N, SEED0 + 1, args.boxes, True, args.faithful_cap)
        cpu = {"value": round(texels / (t1 - t0) / 1e6, 3), "unit": "Mtexels/s", "cores": 4, "kind": "port",
               "cores_note": "MinMaxHierarchy on 4 threads (src/MinMaxHierarchy.cpp:56-66), create() on 1",
               "host": hc,
               "sample": f"one full {N}^2 build: MinMaxHierarchy on 4 threads + create() single-threaded with the "
                         f"hash-table mergeLevel (word-identical to the linear search), {t1 - t0:.2f} s",
               "words_equal_gpu": words_equal,
               "faithful_create": {
                   "1024^2_plane_32_boxes": {"s": None if f0_s is None else round(f0_s, 3), "words": f0_words,
                                             "Mtexels_per_s": None if not f0_s else round(1024 * 1024 / f0_s / 1e6, 3)},
                   f"{N}^2": {"s": f">{args.faithful_cap:.0f}" if f1_s is None else round(f1_s, 2),
                              "cap_s": args.faithful_cap},
                   "note": "the reference's linear-search mergeLevel (src/CompressedShadowUtil.h:154-182), "
                           "1 thread, create() only (pyramid excluded)"},
               "lookup_G_per_s": round(sample / (t3 - t2) / 1e9, 4), "lookup_threads": threads,
               "lookup_G_per_s_1thread": round(2_000_000 / (t5 - t4) / 1e9, 4),
               "lookup_sample": f"traverse.cs transcription over all {sample} queries on {threads} threads "
                                f"({t3 - t2:.2f} s) and the first 2,000,000 on 1 thread ({t5 - t4:.2f} s)"}

    out = {
        "metric": METRIC,
        "value": round(build_rate, 1),
        "unit": "Mtexels/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(statistics.mean(step_ms), 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32 compares, u32 DAG",
        "data": "synthetic (device-generated depth map and G-buffer queries)",
        "config": {"workload": f"{N}x{N} depth map (plane + {args.boxes} boxes + 4-octave noise), "
                               f"{nq} G-buffer lookups ({args.width}x{args.height} x 2)",
                   "N": N, "zTileNum": 1, "queries": nq, "dag_words": words},
        "host_input": host_input,
        "headline_check": check,
        "c0_1024": c0,
        "build_ms_mean": round(statistics.mean(build_ms), 3),
        "build_ms_p50": round(pct(build_ms, 50), 3),
        "build_ms_p99": round(pct(build_ms, 99), 3),
        "lookup_G_per_s": round(lookup_rate, 3),
        "lookup_ms_p50": round(pct(lookup_ms, 50), 3),
        "lookup_ms_p99": round(pct(lookup_ms, 99), 3),
        "lookup_top_table": {"setting": top_set, "levels": top_levels,
                             "tune_ms": {str(k): round(v, 4) for k, v in top_ms.items()},
                             "container_ms_p50": round(pct(container_ms, 50), 3),
                             "build_top_ms": round(prof["build_top"][0] / prof_steps, 4) if "build_top" in prof else 0.0,
                             "lookup_G_per_s_incl_table": round(
                                 nq / ((pct(lookup_ms, 50) + (prof["build_top"][0] / prof_steps if "build_top" in prof
                                                                else 0.0)) * 1e-3) / 1e9, 3),
                             "note": "copyToGPU (combineDAGs, grid, top table) between build and lookup, GPU "
                                     "events; not in build_ms or lookup_ms.  The inclusive rate counts the table's "
                                     "build (k_build_top, once per container) with one evaluate"},
        "roofline": roofline,
        "pyramid_roofline": pyramid_roofline,
        "lookup_roofline": lookup_roofline,
        "device_copy_GBs": round(copy_gbs, 1),
        "kernel_ms_per_step": {k: round(v[0] / prof_steps, 4) for k, v in prof.items()},
        "tiled_65536": tiled,
        "batched_256_maps": batched,
        "serving": serving,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
