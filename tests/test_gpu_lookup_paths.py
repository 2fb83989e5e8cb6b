"""The lookups' dispatch: how a light matrix is applied (identity, affine, full product) with finite
and non-finite positions, PCF windows within, across and beyond 8 x 8 blocks and the grid's border,
and round-robin DAG sets whose groups do not divide over the XCDs.  Results are whole numbers or
exact fractions, so every compare is for equality.  Needs a GPU."""
import numpy as np
import pytest

import cpvs_amd as cp
import oracle as O

pytestmark = pytest.mark.gpu
SEED0 = 0x43505653
N = 128


def _say(*a):
    print("[case]", *a, flush=True)


def _container(D):
    c = cp.CompressedShadowContainer(cp.CompressedShadow.create(cp.MinMaxHierarchy(D)))
    c.copyToGPU()
    return c


def _special():
    """Positions with infinities, NaN, huge and tiny values and signed zeros in every coordinate."""
    v = np.array([0.0, -0.0, 0.25, -1.0, 1.0, 3e38, -3e38, 1e-45, np.inf, -np.inf, np.nan], np.float32)
    g = np.stack(np.meshgrid(v, v, v, indexing="ij"), -1).reshape(-1, 3)
    return np.concatenate([g, np.ones((len(g), 1), np.float32)], 1)


def _np_paths(q, m, R):
    """traverse.cs's path in float32 steps: the product in column order, the divide, the quantisation,
    out-of-range clamped and NaN 0."""
    f = np.float32
    with np.errstate(all="ignore"):
        r = [((m[c, 0] * q[:, 0] + m[c, 1] * q[:, 1]) + m[c, 2] * q[:, 2]) + m[c, 3] for c in range(4)]
        p = [((r[c] / r[3]) + f(1.0)) * f(0.5) * f(R - 1) for c in range(3)]
        p = [np.where(v > 0, np.minimum(v, f(R - 1)), f(0)) for v in p]
    return [v.astype(np.int64) for v in p]


def _matrix(kind):
    m = np.eye(4, dtype=np.float32)
    if kind == "negzero":
        m[m == 0] = -0.0
    elif kind == "affine":
        m[:3] = [[0.7, -0.2, 0.1, 0.05], [0.3, 0.9, -0.15, -0.1], [-0.1, 0.25, 0.8, 0.2]]
    elif kind == "full":
        m[:] = [[0.7, -0.2, 0.1, 0.05], [0.3, 0.9, -0.15, -0.1], [-0.1, 0.25, 0.8, 0.2], [0.1, -0.2, 0.3, 1.5]]
    elif kind == "w2":
        m[3, 3] = 2.0
    return m


@pytest.mark.parametrize("kind", ["none", "identity", "negzero", "affine", "full", "w2"])
@pytest.mark.parametrize("stride", [3, 4])
def test_projections_with_special_positions(ctx, kind, stride):
    _say("projection", kind, stride)
    D = O.gen_depth(N, SEED0 + 5, 6, True)
    rng = np.random.default_rng(3)
    q = np.concatenate([_special(), np.concatenate([rng.uniform(-1.2, 1.2, (3001, 3)), np.ones((3001, 1))], 1)])
    q = np.ascontiguousarray(q, np.float32)
    m = _matrix("identity" if kind == "none" else kind)
    want = O.brute_visible(D, 1, *_np_paths(q, m, N))
    c = _container(D)
    got = c.evaluate(cp.DeviceArray.from_numpy(q[:, :stride]), None if kind == "none" else m).numpy()
    assert np.array_equal(got, want.astype(np.uint8))
    c.close()


@pytest.mark.parametrize("f", [2, 3, 8, 9, 16, 17, 64])
def test_pcf_windows(ctx, f):
    """Every window position against a block's and the grid's border (one row of paths per axis)."""
    _say("pcf", f)
    D = O.gen_depth(N, SEED0 + 6, 6, True)
    a = np.arange(N)
    p = np.concatenate([np.stack([a, np.full(N, 61), a], 1), np.stack([np.full(N, 61), a, N - 1 - a], 1),
                        np.stack([a, a, (D[a, a] * N).astype(int).clip(0, N - 1)], 1),
                        np.stack([N - 1 - a, a, (D[a, N - 1 - a] * N).astype(int).clip(0, N - 1)], 1)])
    q = ((p + 0.5) / (N - 1) * 2 - 1).clip(-1, 1).astype(np.float32)
    p = np.stack(_np_paths(q, np.eye(4, dtype=np.float32), N), 1)
    lo, lit = -((f - 1) // 2), np.zeros(len(p), np.int64)
    for dy in range(f):
        for dx in range(f):
            lit += O.brute_visible(D, 1, np.clip(p[:, 0] + lo + dx, 0, N - 1), np.clip(p[:, 1] + lo + dy, 0, N - 1), p[:, 2])
    c = _container(D)
    c.setFilterSize(f)
    got = c.evaluate_pcf(cp.DeviceArray.from_numpy(q)).numpy()
    assert np.array_equal(got, lit.astype(np.float32) / np.float32(f * f))
    c.close()


@pytest.mark.parametrize("dags,count", [(1, 1), (1, 4097), (3, 64), (16, 16 * 64), (17, 20011), (48, 9999), (130, 70001)])
def test_round_robin_tiles(ctx, dags, count):
    _say("round robin", dags, count)
    D = [O.gen_depth(32 << (i % 2), SEED0 + 20 + i, 1 + i % 3, True) for i in range(min(dags, 7))]
    sh = [cp.CompressedShadow.create(cp.MinMaxHierarchy(d)) for d in D]
    some = [sh[i % len(sh)] for i in range(dags)]
    q = np.random.default_rng(dags).uniform(-1, 1, (count, 3)).astype(np.float32)
    got = cp.DagSet(some).evaluate(cp.DeviceArray.from_numpy(q)).numpy()
    want = np.zeros(count, np.uint8)
    for i in range(dags):
        d = D[i % len(D)]
        mine = q[i::dags]
        want[i::dags] = O.brute_visible(d, 1, *_np_paths(mine, np.eye(4, dtype=np.float32), d.shape[0]))
    assert np.array_equal(got, want)
    for s in sh:
        s.close()


@pytest.mark.parametrize("leafmasks", [1, 0])
@pytest.mark.parametrize("N,length", [(8, 1), (16, 2), (64, 1), (64, 2), (128, 4), (256, 1), (256, 4)])
@pytest.mark.parametrize("top", [0, 1, -1])
def test_links_of_container_dags(ctx, N, length, top, leafmasks):
    """Lookups through the container's links, over the words copied with them: cells of one word (empty
    and full z-tiles) beside cells of many, below, at and above one tile of words."""
    _say("links", N, length, top, leafmasks)
    ctx.set_leafmasks(bool(leafmasks))
    try:
        c = cp.CompressedShadowContainer(length)
        words, order = [], {}
        for y in range(length):
            for x in range(length):
                D = O.gen_depth(N, SEED0 + 30 + y * length + x, 3, True)
                for z in range(length):
                    sh = cp.CompressedShadow.create(cp.MinMaxHierarchy(D), z, length)
                    order[(z, y, x)] = sh.getDAG()
                    n = sh.getNumLevels()
                    c.set(sh, x, y, z)
        words = [order[k] for k in sorted(order)]
        c.setTopLevels(top)
        c.moveToGPU()
        w, grid = c.words_and_grid()
        assert np.array_equal(w, np.concatenate(words))
        assert np.array_equal(grid, O.top_level_grid(words))
        q = np.random.default_rng(N + length).uniform(-1, 1, (20011, 4)).astype(np.float32)
        got = c.evaluate(cp.DeviceArray.from_numpy(q)).numpy()
        gl = length.bit_length() - 1
        px = _np_paths(q, np.eye(4, dtype=np.float32), N * length)
        want = np.zeros(len(q), np.uint8)
        for y in range(length):
            for x in range(length):
                D = O.gen_depth(N, SEED0 + 30 + y * length + x, 3, True)
                here = (px[0] // N == x) & (px[1] // N == y)
                want[here] = O.brute_visible(D, length, px[0][here] % N, px[1][here] % N, px[2][here])
        assert (n, gl) == c.info()[:2] and np.array_equal(got, want)
        c.close()
    finally:
        ctx.set_leafmasks(True)
