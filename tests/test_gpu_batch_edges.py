"""Batches around the changes of rule: few queries for their triangles (the FP32 nodes) and
many (the oriented ones), and as many meshes as the first levels' one-block launch takes,
one more, and so many that the tree is one level of it.  Answers equal the brute force, replay
after replay.
"""
import numpy as np
import pytest
import torch

import gpurt
from gpurt import _lib
from gpurt import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(ctx, dev, meshes, **kw):
    dm = [{k: torch.from_numpy(v).to(dev) for k, v in m.items()} for m in meshes]
    batch = gpurt.Batch(ctx, dm, **kw)
    for _ in range(3):
        res = batch.run()
        torch.cuda.synchronize()
        for i, (h, r) in enumerate(zip(meshes, res)):
            ep, ept, ed, _ = O.cpq_brute_f32(h["verts"], h["tris"], h["queries"])
            assert np.array_equal(r["q_prim"].cpu().numpy(), ep), i
            assert np.array_equal(r["q_dist"].cpu().numpy(), ed), i
            assert np.array_equal(r["q_pt"].cpu().numpy(), ept), i
            rp, rt, _ = O.ray_closest_brute_f32(h["verts"], h["tris"], h["rays"])
            assert np.array_equal(r["r_prim"].cpu().numpy(), rp), i
            assert np.array_equal(r["r_t"].cpu().numpy(), rt), i
            for v in r.values():
                v.zero_()


def _mesh(level, nq, nr, seed):
    rng = np.random.default_rng(seed)
    v, f = W.displaced_icosphere(level, rng)
    rays = W.pack_rays(rng.uniform(-2, 2, (nr, 3)), W.random_dirs(rng, nr), 1e-5, 1e7)
    return {"verts": v.astype(np.float32), "tris": f.astype(np.int32),
            "queries": rng.uniform(-1.5, 1.5, (nq, 3)).astype(np.float32), "rays": rays}


@pytest.mark.parametrize("nq", [1, 319, 320, 321, 2000])
def test_batch_node_choice_by_queries(ctx, dev, nq):
    """1,280 triangles in all: from 320 queries on the oriented nodes are made."""
    _check(ctx, dev, [_mesh(2, 0 if k else nq, 50, k) for k in range(4)])


@pytest.mark.parametrize("n,width", [(1, 2), (64, 4), (65, 4), (255, 8), (256, 2), (257, 4), (300, 8)])
def test_batch_mesh_counts(ctx, dev, n, width):
    print("batch of", n, "meshes, width", width, flush=True)
    _check(ctx, dev, [_mesh(k % 3, 1 + k % 70, 1 + k % 30, k) for k in range(n)], node_width=width)


@pytest.mark.parametrize("mode", ["auto", "fixed", "atomic"])
def test_batch_meshes_may_share_a_vertex_gradient(dev, mode):
    """Two meshes whose g_verts is one buffer: it gets both meshes' gradients.  In the fixed
    order each mesh adds one total per vertex, so it is exactly their rounded sum; with atomics
    two FP32 sums of up to c terms of at most 1 differ by at most 2 c^2 2^-24."""
    ctx = gpurt.Context(0, vertex_sums=mode)
    n = 110_000  # with 2 meshes more than 600,000 terms
    meshes = [_mesh(4, n, 1, 3), _mesh(4, n, 1, 3)]
    q = W.surface_samples(meshes[1]["verts"].astype(np.float64), meshes[1]["tris"], np.random.default_rng(8), n, 0.02)
    meshes[1]["queries"] = q.astype(np.float32)
    batch = gpurt.Batch(ctx, [{k: torch.from_numpy(v).to(dev) for k, v in m.items()} for m in meshes])
    own = batch.enable_backward()
    res = batch.run()
    batch.backward()
    torch.cuda.synchronize()
    c = sum(np.bincount(m["tris"][r["q_prim"].cpu().numpy()].ravel(), minlength=len(m["verts"])) for m, r in
            zip(meshes, res)).max() + 2
    want = own[0]["g_verts"] + own[1]["g_verts"]
    both = own[0]["g_verts"]
    batch._garr[1].g_verts = both.data_ptr()
    assert _lib.load().gpurt_batch_set_grads(batch._h, batch._garr) == 0
    for _ in range(10):
        batch.backward()
        torch.cuda.synchronize()
        if mode == "atomic":
            assert float((both - want).abs().max()) <= 2.0 * c * c * 2.0**-24
        else:
            assert torch.equal(both, want)
    batch.close()
    ctx.close()
