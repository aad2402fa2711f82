"""Closest points through the oriented nodes (4-wide, the default format): ids, points and
distances equal the FP32 nodes' on the same mesh bit for bit, and the oracle's brute force,
on the meshes where a node's frame or byte grid can go wrong -- sizes around the ones at
which a node is made by 4 lanes, 16 lanes or a wave or keeps its axis-aligned boxes, flat and
needle-shaped and coincident triangles, normals along the axes and opposite to each other,
far-away and huge and tiny coordinates -- and after a refit.
"""
import numpy as np
import pytest
import torch

import gpurt
from gpurt import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _grid(n, m, f):
    x, y = np.meshgrid(np.linspace(-1, 1, n + 1), np.linspace(-1, 1, m + 1), indexing="ij")
    v = f(x.ravel(), y.ravel())
    i = (np.arange(n)[:, None] * (m + 1) + np.arange(m)[None, :]).ravel()
    t = np.concatenate([np.stack([i, i + m + 1, i + 1], 1), np.stack([i + 1, i + m + 1, i + m + 2], 1)])
    return v, t


def _mesh(kind):
    rng = np.random.default_rng(len(kind))
    if kind.startswith("sphere"):
        v, f = W.displaced_icosphere(int(kind[-1]), rng)
    elif kind == "plane":  # one normal, boxes without thickness
        v, f = _grid(37, 29, lambda x, y: np.stack([x, y, 0.3 * x - 0.7 * y], 1))
    elif kind == "axis_planes":  # normals along the axes, both ways round
        v, f = [], []
        for a in range(3):
            g, t = _grid(9, 9, lambda x, y: np.roll(np.stack([x, y, np.zeros_like(x)], 1), a, 1))
            f += [t + sum(map(len, v)), t[:, ::-1] + sum(map(len, v))]
            v.append(g)
        v, f = np.concatenate(v), np.concatenate(f)
    elif kind == "needles":
        c = rng.uniform(-1, 1, (700, 1, 3))
        d = W.random_dirs(rng, 700)[:, None]
        v = (c + d * np.array([-0.5, 0.0, 0.5])[None, :, None] + rng.normal(0, 1e-6, (700, 3, 3))).reshape(-1, 3)
        f = np.arange(2100).reshape(-1, 3)
    elif kind == "points":  # triangles without area
        v = np.repeat(rng.uniform(-1, 1, (500, 1, 3)), 3, 1).reshape(-1, 3)
        f = np.arange(1500).reshape(-1, 3)
    elif kind == "one_place":  # all triangles the same
        v, f = np.array([[0.1, 0.2, 0.3], [0.2, 0.2, 0.3], [0.1, 0.3, 0.35]]), np.tile([[0, 1, 2]], (300, 1))
    else:  # random triangles of mixed winding
        n = int(kind.split("_")[1])
        v = (rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0, 0.05, (n, 3, 3))).reshape(-1, 3)
        f = np.arange(3 * n).reshape(-1, 3)
    return v, f.astype(np.int32)


def _queries(V, F, n, seed):
    rng = np.random.default_rng(seed)
    lo, hi = V.min(0).astype(np.float64), V.max(0).astype(np.float64)
    ext = (hi - lo).max()
    near = W.surface_samples(V.astype(np.float64), F, rng, n // 2, 0.01 * ext)
    box = (lo + hi) / 2 + rng.uniform(-1.5, 1.5, (n // 4, 3)) * ext
    far = (lo + hi) / 2 + W.random_dirs(rng, n - n // 2 - n // 4) * ext * 30.0
    at = V[F[rng.integers(0, F.shape[0], 16)]].reshape(-1, 3)  # on vertices: ties
    return np.concatenate([near, box, far, at]).astype(np.float32)


def _same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(x.cpu().numpy(), y.cpu().numpy())


@pytest.mark.parametrize("tsize,leaf", [(0, 4), (7, 4), (0, 1), (5, 8)])
@pytest.mark.parametrize("kind", ["random_1", "random_3", "random_17", "random_64", "random_65", "random_4096",
                                  "random_4097", "random_9001", "sphere4", "plane", "axis_planes", "needles", "points",
                                  "one_place"])
def test_oriented_nodes_answer_as_fp32_nodes(ctx, dev, kind, tsize, leaf):
    print("oriented", kind, tsize, leaf, flush=True)
    v, F = _mesh(kind)
    for scale, shift in ((1.0, 0.0), (1.0, 50.0), (1e-15, 0.0), (1e12, 0.0)):
        V = ((v + shift) * scale).astype(np.float32)
        Q = _queries(V, F, 600, 5)
        got = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev), treelet_size=tsize, leaf_size=leaf)
        assert got.info()["cpq_node_bytes"] == 64 and got.info()["node_format"] == 3
        ref = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev), treelet_size=tsize, leaf_size=leaf, node_format=1)
        a, b = got.closest_point(_t(Q, dev)), ref.closest_point(_t(Q, dev))
        _same(a, b)
        if scale == 1.0:
            ep, ept, ed, _ = O.cpq_brute_f32(V, F, Q)
            assert np.array_equal(a[0].cpu().numpy(), ep) and np.array_equal(a[2].cpu().numpy(), ed)
            assert np.array_equal(a[1].cpu().numpy(), ept)


@pytest.mark.parametrize("big", [1e25, 3e38])
def test_oriented_nodes_at_overflowing_coordinates(ctx, dev, big):
    """Distances whose squares overflow, and boxes that do: every triangle is a candidate at
    an infinite distance, as with the FP32 nodes."""
    v, F = _mesh("random_65")
    V = v.astype(np.float32)
    V[F[::7].ravel()] *= np.float32(big)
    V = np.clip(V, -3.4e38, 3.4e38).astype(np.float32)
    Q = np.concatenate([np.random.default_rng(1).uniform(-1, 1, (200, 3)), V[:40],
                        [[3e38, -3e38, 3e38], [1e30, 0, 0]]]).astype(np.float32)
    got = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev)).closest_point(_t(Q, dev))
    ref = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev), node_format=1).closest_point(_t(Q, dev))
    assert np.array_equal(got[0].cpu().numpy(), ref[0].cpu().numpy())
    assert np.array_equal(got[2].cpu().numpy(), ref[2].cpu().numpy())


@pytest.mark.parametrize("tsize", [0, 7])
def test_oriented_nodes_after_refit(ctx, dev, tsize):
    v, F = W.displaced_icosphere(4, np.random.default_rng(2))
    V = v.astype(np.float32)
    tv = _t(V, dev)
    bvh = gpurt.Bvh(ctx, tv, _t(F.astype(np.int32), dev), treelet_size=tsize)
    rng = np.random.default_rng(3)
    for k in range(3):
        a = np.linalg.qr(rng.normal(size=(3, 3)))[0]  # every normal turns
        V2 = ((v * (1.0 + 0.2 * k)) @ a + rng.normal(0, 0.002, v.shape)).astype(np.float32)
        bvh.refit(_t(V2, dev))
        Q = _queries(V2, F.astype(np.int32), 500, k)
        p, pt, d, _ = bvh.closest_point(_t(Q, dev))
        ep, ept, ed, _ = O.cpq_brute_f32(V2, F.astype(np.int32), Q)
        assert np.array_equal(p.cpu().numpy(), ep) and np.array_equal(d.cpu().numpy(), ed)
        assert np.array_equal(pt.cpu().numpy(), ept)
