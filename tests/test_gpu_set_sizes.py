"""The size of a query set chooses the launch's lanes (a wave per query, down to four lanes
and one lane per query) and whether the work queues are used at all.  The answers of a set
do not depend on it: every prefix of a large set answers like the large set does, in
particular right after a launch that left the queue counters used.  The sizes lie around the
changes of rule on a device of 256 CUs.
"""
import numpy as np
import pytest
import torch

import gpurt
from gpurt import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

N = 600_000
SIZES = [1, 2, 63, 64, 65, 2047, 2048, 2049, 4095, 4096, 4097, 32768, 32769, 65536, 65537, 262143, 262144, 262145,
         458751, 458752, 458753]


@pytest.fixture(scope="module")
def scene(ctx, dev):
    rng = np.random.default_rng(11)
    v, f = W.displaced_icosphere(5, rng)
    V, F = v.astype(np.float32), f.astype(np.int32)
    bvh = gpurt.Bvh(ctx, torch.from_numpy(V).to(dev), torch.from_numpy(F).to(dev))
    tlas = gpurt.Tlas(ctx, [(bvh, np.eye(3, 4), 7)])
    q = np.where(rng.random((N, 1)) < 0.9, W.surface_samples(v, f, rng, N, 0.05), rng.uniform(-2, 2, (N, 3)))
    o = rng.uniform(-2, 2, (N, 3))
    d = W.random_dirs(rng, N)
    rays = np.concatenate([o, np.zeros((N, 1)), d, np.full((N, 1), 1e30)], 1).astype(np.float32)
    q = q.astype(np.float32)
    tq, tr = torch.from_numpy(q).to(dev), torch.from_numpy(rays).to(dev)
    run = {"points": lambda n: bvh.closest_point(tq[:n])[:3],
           "closest": lambda n: bvh.trace_closest(tr[:n])[:2],
           "any": lambda n: (bvh.trace_any(tr[:n]),),
           "tlas": lambda n: tlas.trace_closest(tr[:n])[:3]}
    return V, F, q, rays, {k: (f, [x.clone() for x in f(N)]) for k, f in run.items()}


@pytest.mark.parametrize("kind", ["points", "closest", "any", "tlas"])
def test_prefix_of_a_set_answers_like_the_set(scene, kind):
    run, full = scene[4][kind]
    for n in SIZES:
        got = run(n)
        assert len(got) == len(full)
        for a, b in zip(got, full):
            assert torch.equal(a, b[:n]), n
        for a, b in zip(run(N), full):  # and leaves the queue counters used
            assert torch.equal(a, b), n


def test_large_set_against_brute_force(scene):
    V, F, q, rays, out = scene
    pick = np.random.default_rng(1).integers(0, N, 400)
    p, pt, d, _ = O.cpq_brute_f32(V, F, q[pick])
    got = [x.cpu().numpy()[pick] for x in out["points"][1]]
    assert np.array_equal(got[0], p) and np.array_equal(got[1], pt) and np.array_equal(got[2], d)
