"""Handle lifetime: destruction is stream-ordered (a BVH destroyed while a query that
reads it is still running on another stream is freed only after that query), a context
destroyed before its handles releases their device memory and leaves them safe to
destroy, and a process that exits with objects still open exits cleanly."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest
import torch

import gpurt
from gpurt import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def test_destroy_while_a_query_runs_on_another_stream(ctx, dev):
    w = W.rays_scene(n_rays=1 << 20, grid=301, n_spheres=16)
    V, F, R = w["verts"], w["tris"], w["rays"]
    sub = np.arange(0, R.shape[0], 512)
    ep, et, _ = O.CpuBvh(V, F).trace_closest(R[sub])
    tr = _t(R, dev)
    side = torch.cuda.Stream(dev)
    for _ in range(3):
        bvh = gpurt.Bvh(ctx, _t(V, dev), _t(F, dev))
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            prim, t, _ = bvh.trace_closest(tr)
            for _ in range(3):  # keep the stream busy well past the destroy below
                bvh.trace_closest(tr)
        bvh.close()  # returns at once; the memory is released after the queries
        # reuse the released memory on the default stream while the side stream runs
        other = gpurt.Bvh(ctx, _t(V * np.float32(2.0), dev), _t(F, dev))
        side.synchronize()
        assert np.array_equal(prim.cpu().numpy()[sub], ep) and np.array_equal(t.cpu().numpy()[sub], et)
        other.close()


def test_context_destroyed_before_its_handles(dev):
    c2 = gpurt.Context(0)
    w = W.cpq_small(n_queries=64)
    V, F = _t(w["verts"], dev), _t(w["tris"], dev)
    bvh = gpurt.Bvh(c2, V, F)
    tlas = gpurt.Tlas(c2, [(bvh, np.eye(3, 4))])
    prim, _, _, _ = bvh.closest_point(_t(w["queries"], dev))
    torch.cuda.synchronize()
    c2.close()  # releases the BVH's and TLAS's device memory
    tlas.close()  # host part only
    bvh.close()
    assert prim.cpu().numpy().min() >= 0


def test_process_exits_cleanly_with_objects_open():
    code = r"""
import sys, numpy as np, torch
sys.path[:0] = [sys.argv[1], sys.argv[2]]
import gpurt
from gpurt import workloads as W
dev = torch.device("cuda", 0)
ctx = gpurt.Context(0)
w = W.rays_scene(n_rays=4096, grid=41, n_spheres=2)
V, F = torch.from_numpy(w["verts"]).to(dev), torch.from_numpy(w["tris"]).to(dev)
bvh = gpurt.Bvh(ctx, V, F)
tlas = gpurt.Tlas(ctx, [(bvh, np.eye(3, 4))])
rays = torch.from_numpy(w["rays"]).to(dev)
s = torch.cuda.Stream(dev)
with torch.cuda.stream(s):
    bvh.trace_closest(rays)
    tlas.trace_any(rays)
batch = gpurt.Batch(ctx, [{"verts": V, "tris": F, "rays": rays}])
batch.run()
print("ok", flush=True)
# exit with everything open and queries in flight
"""
    r = subprocess.run([sys.executable, "-c", code, os.path.join(ROOT, "gpu-rt_amd"), ROOT],
                       capture_output=True, text=True, timeout=240)
    print(r.stdout, r.stderr[-2000:])
    assert r.returncode == 0 and "ok" in r.stdout


def _sleep(stream, seconds):
    """A spinning kernel of about that time on the stream."""
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    cycles = 1_000_000
    with torch.cuda.stream(stream):
        torch.cuda._sleep(cycles)
        a.record(stream)
        torch.cuda._sleep(cycles)
        b.record(stream)
        b.synchronize()
        torch.cuda._sleep(int(cycles * seconds * 1e3 / a.elapsed_time(b)))


def _soup(n, dev):
    g = torch.Generator(device=dev).manual_seed(1)
    c = torch.rand(n, 1, 3, generator=g, device=dev)
    v = (c + 0.01 * torch.rand(n, 3, 3, generator=g, device=dev)).reshape(-1, 3).contiguous()
    return v, torch.arange(3 * n, device=dev, dtype=torch.int32).reshape(-1, 3)


@pytest.fixture
def many_bvhs(dev):
    """A context and BVHs whose memory together is more than the context keeps idle (a
    sixteenth of the device's)."""
    V, F = _soup(2_000_000, dev)
    ctx = gpurt.Context(0)
    free0, total = torch.cuda.mem_get_info(dev)
    bvhs = []
    while len(bvhs) < 400 and free0 - torch.cuda.mem_get_info(dev)[0] < total / 16 + (4 << 30):
        bvhs += [gpurt.Bvh(ctx, V, F) for _ in range(8)]
    yield V[:4096].contiguous(), bvhs
    ctx.close()
    torch.cuda.synchronize()
    # given back with the context
    assert torch.cuda.mem_get_info(dev)[0] > free0 - (1 << 30)


def test_destroy_beyond_the_idle_limit_does_not_wait(dev, many_bvhs):
    """Destroying them while a query on the first is still to run waits for nothing, and the
    query's answer is whole."""
    Q, bvhs = many_bvhs
    busy, done = torch.cuda.Stream(dev), torch.cuda.Event()
    want = bvhs[0].closest_point(Q)
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        bvhs[0].closest_point(Q)
        _sleep(busy, 0.5)
        got = bvhs[0].closest_point(Q)
        done.record(busy)
    for b in bvhs:
        b.close()
    assert not done.query(), "a destroy waited for the query"
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_destroy_beyond_the_idle_limit_while_another_thread_captures(dev, many_bvhs):
    """Destroying them while a stream is captured in HIP's global mode leaves the capture whole."""
    _, bvhs = many_bvhs
    x = torch.arange(1024, dtype=torch.float32, device=dev)
    y = torch.zeros_like(x)
    t = threading.Thread(target=lambda: [b.close() for b in bvhs])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="global"):
        torch.add(x, 1.0, out=y)
        t.start()
        t.join(60)
        torch.mul(y, 2.0, out=y)
    for _ in range(2):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, (x + 1.0) * 2.0)
