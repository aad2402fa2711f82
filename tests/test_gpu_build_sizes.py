"""The builder at the sizes where its passes change: one-block and multi-block sorts (8192
pairs), chunks of 256 leaves and the aligned blocks above them (powers of four), trees
deeper than the launches for their size, and memory that goes from one BVH to the next.

Every size is checked against the mesh itself: the packed order is the oracle's Morton
order (stable, so equal codes stay in triangle order), a leaf child's box is exactly its
triangles' bounds and an inner child's box exactly the union of that child's own boxes
(minima and maxima round nothing; both sides carry the same inflation), so each binary
node's box is the bottom-up one whichever pass made it.
"""
import numpy as np
import pytest
import torch

import gpurt
from gpurt import _lib
from gpurt import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LEAF = np.uint32(0x80000000)
EMPTY = np.uint32(0xFFFFFFFF)


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _soup(n, seed, dup=0.0):
    """n random triangles; a share `dup` of them at one place (equal Morton codes)."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (n, 1, 3))
    c[rng.uniform(size=n) < dup] = 0.25
    v = (c + rng.normal(0, 0.02, (n, 3, 3))).astype(np.float32).reshape(-1, 3)
    return v, np.arange(3 * n, dtype=np.int32).reshape(-1, 3)


def _check(bvh, V, F, morton_order=True):
    info = bvh.info()
    w, nt = info["node_width"], info["n_tris"]
    ex = {k: v.cpu().numpy() for k, v in bvh.export().items() if v is not None}
    nodes = ex["nodes"].view(np.float32)
    lo = np.stack([nodes[:, a * w:(a + 1) * w] for a in range(3)], -1)
    hi = np.stack([nodes[:, (3 + a) * w:(4 + a) * w] for a in range(3)], -1)
    child = nodes[:, 6 * w:7 * w].view(np.uint32)
    count = nodes[:, 7 * w:8 * w].view(np.uint32)
    tri = ex["tris"].reshape(nt, 3, 4)[:, :, :3]
    order = ex["leaf_order"]
    if morton_order:
        assert np.array_equal(order, O.CpuBvh(V, F, 4).order())
    assert np.array_equal(np.sort(order), np.arange(nt))
    assert np.array_equal(tri, V[F[order]])
    pad = np.float32(np.abs(V[F]).max()) * np.float32(2.0 ** -18)
    leaf = (child != EMPTY) & ((child & LEAF) != 0)
    inner = (child & LEAF) == 0
    # leaves: disjoint ranges that cover the triangles, boxes from them
    first, cnt = (child & 0x0FFFFFFF)[leaf].astype(np.int64), (((child >> 28) & 7) + 1)[leaf].astype(np.int64)
    assert np.array_equal(count[leaf], cnt)
    cover = np.zeros(nt + 1, np.int64)
    np.add.at(cover, first, 1)
    np.add.at(cover, first + cnt, -1)
    assert (np.cumsum(cover)[:nt] == 1).all()
    tlo, thi = tri.min(1), tri.max(1)
    for k in range(int(cnt.max())):
        on = k < cnt
        at = (first + k)[on]
        if k == 0:
            blo, bhi = tlo[first].copy(), thi[first].copy()
        else:
            blo[on] = np.minimum(blo[on], tlo[at])
            bhi[on] = np.maximum(bhi[on], thi[at])
    assert np.array_equal(lo[leaf], blo - pad) and np.array_equal(hi[leaf], bhi + pad)
    # inner children: the union of their own boxes, the sum of their counts
    if inner.any():
        c = child[inner].astype(np.int64)
        assert np.array_equal(np.sort(c), np.arange(1, child.shape[0]))
        assert np.array_equal(lo[inner], lo[c].min(1)) and np.array_equal(hi[inner], hi[c].max(1))
        assert np.array_equal(count[inner], count[c].sum(1))
    assert count[0].sum() == nt
    return info


@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 256, 257, 511, 1024, 1025, 4095, 4097, 8191, 8192, 8193, 16384, 65537])
def test_build_at_pass_edges(ctx, dev, n):
    print("build", n, flush=True)
    V, F = _soup(n, n, dup=0.3 if n % 2 else 0.0)
    _check(gpurt.Bvh(ctx, _t(V, dev), _t(F, dev)), V, F)


@pytest.mark.parametrize("n,leaf,tsize", [(257, 1, 5), (4097, 8, 7), (8193, 4, 7), (20000, 2, 6)])
def test_treelet_build_at_pass_edges(ctx, dev, n, leaf, tsize):
    print("treelets", n, leaf, tsize, flush=True)
    V, F = _soup(n, n + 1, dup=0.1)
    _check(gpurt.Bvh(ctx, _t(V, dev), _t(F, dev), leaf_size=leaf, treelet_size=tsize), V, F, morton_order=False)


@pytest.mark.parametrize("width", [2, 4, 8])
def test_tree_deeper_than_its_launches(ctx, dev, width):
    """A few triangles at halving distances along each axis from a cluster of equal codes:
    one binary level per triangle on the way to the cluster."""
    n = 8000
    c = [np.zeros(3)]
    for j in range(11):
        for a in range(3):
            p = np.zeros(3)
            p[a] = 2.0 ** -j
            c.append(p)
    c = np.concatenate([np.array(c), np.zeros((n, 3))])
    rng = np.random.default_rng(3)
    V = (c[:, None] + rng.uniform(0, 1e-4, (c.shape[0], 3, 3))).astype(np.float32).reshape(-1, 3)
    F = np.arange(V.shape[0], dtype=np.int32).reshape(-1, 3)
    bvh = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev), node_width=width)
    info = _check(bvh, V, F)
    # (the launches enqueued for 13 bits of triangles at each width)
    assert info["depth"] > {2: 15, 4: 12, 8: 8}[width]
    o = rng.uniform(-0.5, 1.5, (512, 3))
    R = W.pack_rays(o, W.random_dirs(rng, 512), 1e-5, 1e7)
    prim, t, _ = bvh.trace_closest(_t(R, dev))
    ep, et, _ = O.ray_closest_brute_f32(V, F, R)
    assert np.array_equal(prim.cpu().numpy(), ep) and np.array_equal(t.cpu().numpy(), et)


def test_memory_of_closed_bvhs_is_reused_in_order(dev):
    """BVHs built, queried and closed on two streams with no host wait of the caller's: a
    block goes to the next build only after the last query of the BVH that had it."""
    ctx = gpurt.Context(0)
    rng = np.random.default_rng(8)
    meshes = [_soup(n, n) for n in (3000, 3100, 9000, 2900)]
    R = [W.pack_rays(rng.uniform(-1, 1, (4096, 3)), W.random_dirs(rng, 4096), 1e-5, 1e7) for _ in meshes]
    exp = [O.ray_closest_brute_f32(V, F, r)[0] for (V, F), r in zip(meshes, R)]
    tm = [(_t(V, dev), _t(F, dev), _t(r, dev)) for (V, F), r in zip(meshes, R)]
    streams = [torch.cuda.Stream(dev), torch.cuda.Stream(dev)]
    torch.cuda.synchronize()
    got = []
    for k in range(24):
        with torch.cuda.stream(streams[k % 2]):
            V, F, r = tm[k % 4]
            bvh = gpurt.Bvh(ctx, V, F)
            got.append(bvh.trace_closest(r)[0])
            bvh.close()
    torch.cuda.synchronize()
    for k, p in enumerate(got):
        assert np.array_equal(p.cpu().numpy(), exp[k % 4]), k
    ctx.close()


def _best_sah(V, F):
    """Least SAH cost of any binary tree over the triangles, one per leaf, without the
    root's own term and over the root's area (1.2 per unit of inner area, 1 per leaf's)."""
    n = F.shape[0]
    t = V[F].astype(np.float64)
    area, cost = np.zeros(1 << n), np.zeros(1 << n)
    for s in range(1, 1 << n):
        p = t[[j for j in range(n) if s >> j & 1]].reshape(-1, 3)
        e = p.max(0) - p.min(0)
        area[s] = 2 * (e[0] * e[1] + e[1] * e[2] + e[0] * e[2])
    for s in range(1, 1 << n):
        low = s & -s
        if s == low:
            cost[s] = area[s]
            continue
        best, p = np.inf, (s - 1) & s
        while p:
            if p & low:
                best = min(best, cost[p] + cost[s ^ p])
            p = (p - 1) & s
        cost[s] = 1.2 * area[s] + best
    full = (1 << n) - 1
    return (cost[full] - 1.2 * area[full]) / area[full]


@pytest.mark.parametrize("tsize", [5, 6, 7])
@pytest.mark.parametrize("n", [3, 4, 5, 6, 7])
def test_treelet_of_the_whole_mesh_is_optimal(ctx, dev, n, tsize):
    """With at most tsize triangles the root's treelet is the whole tree: its topology is the
    best of all (boxes carry an inflation of 2^-18 of the coordinates, under 1e-3 of the
    cost of boxes of about 0.05)."""
    if n > tsize:
        pytest.skip("more triangles than a treelet has leaves")
    for seed in range(4):
        V, F = _soup(n, 100 * n + seed)
        bvh = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev), node_width=2, leaf_size=1, treelet_size=tsize)
        want = _best_sah(V, F)
        assert abs(bvh.info()["sah_cost"] - want) <= 2e-3 * want, (seed, bvh.info()["sah_cost"], want)


@pytest.mark.parametrize("n", [65536, 262143, 262144, 262145, 600_001])
def test_build_at_range_level_edges(ctx, dev, n):
    """Sizes at which the boxes above the 256-node chunks take another level (256 and 1,024
    chunks: a second launch) and the upper nodes' boxes come from them."""
    print("build", n, flush=True)
    V, F = _soup(n, n, dup=0.0)
    _check(gpurt.Bvh(ctx, _t(V, dev), _t(F, dev)), V, F)


def _fractal(n):
    """Soups at 16 halving scales about one point: trees much deeper than their size asks for, of
    many nodes per level all the way down."""
    rng = np.random.default_rng(3)
    c = rng.uniform(-1, 1, (n, 1, 3))
    v = (c + rng.normal(0, 0.02, (n, 3, 3))) * 0.5 ** rng.integers(0, 16, (n, 1, 1))
    return v.astype(np.float32).reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(-1, 3)


@pytest.mark.parametrize("n,width,tsize", [(20_000, 2, 0), (20_000, 2, 5), (20_000, 2, 7), (20_000, 4, 7), (20_000, 8, 7),
                                           (600_000, 2, 0), (600_000, 2, 7), (600_000, 4, 7), (600_000, 8, 0)])
def test_deep_trees_are_built_or_refused(ctx, dev, n, width, tsize):
    """A tree deeper than the supported level count (binary nodes with treelets, 600,000
    triangles) is refused with GPURT_E_UNSUPPORTED, by a plain build and by a batch; any other
    answers as the brute force."""
    print("fractal", n, width, tsize, flush=True)
    V, F = _fractal(n)
    tv, tf = _t(V, dev), _t(F, dev)
    rng = np.random.default_rng(4)
    q = V[3 * rng.integers(0, n, 64)]
    q = (q + 0.01 * np.linalg.norm(q, axis=1, keepdims=True) * rng.normal(size=(64, 3))).astype(np.float32)
    meshes = [{"verts": tv, "tris": tf, "queries": _t(q, dev)}]
    opts = {"node_width": width, "treelet_size": tsize}
    if (n, width, tsize) == (600_000, 2, 7):
        for _ in range(2):
            for build in (lambda: gpurt.Bvh(ctx, tv, tf, **opts), lambda: gpurt.Batch(ctx, meshes, **opts)):
                with pytest.raises(gpurt.GpurtError) as e:
                    build()
                assert e.value.code == _lib.GPURT_E_UNSUPPORTED
        return
    ep, _, ed, _ = O.cpq_brute_f32(V, F, q)
    bvh = gpurt.Bvh(ctx, tv, tf, **opts)
    print("depth", bvh.info()["depth"], flush=True)
    batch = gpurt.Batch(ctx, meshes, **opts)
    r = batch.run()[0]
    for prim, dist in (bvh.closest_point(_t(q, dev))[::2], (r["q_prim"], r["q_dist"])):
        assert np.array_equal(prim.cpu().numpy(), ep) and np.array_equal(dist.cpu().numpy(), ed)
    batch.close()
    bvh.close()
