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


def _two_queues(dev):
    """Two streams whose work runs side by side (streams share the few hardware queues, and
    what is behind a running kernel in its queue waits for it)."""
    busy = torch.cuda.Stream(dev)
    x = torch.zeros(1, device=dev)
    for _ in range(16):
        side = torch.cuda.Stream(dev)
        torch.cuda.synchronize()
        _sleep(busy, 0.1)
        slept = torch.cuda.Event()
        slept.record(busy)
        with torch.cuda.stream(side):
            x.add_(1.0)
        side.synchronize()
        if not slept.query():
            torch.cuda.synchronize()
            return busy, side
    pytest.skip("no two streams run side by side")


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
    query's answer is whole although the next builds take as much memory."""
    Q, bvhs = many_bvhs
    busy, side = _two_queues(dev)
    done = torch.cuda.Event()
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
    V = Q.repeat(300, 1)
    F = torch.arange(3 * (len(V) // 3), device=dev, dtype=torch.int32).reshape(-1, 3)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        others = [gpurt.Bvh(bvhs[0].ctx, V, F) for _ in bvhs]
    torch.cuda.synchronize()
    for b in others:
        b.close()
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


@pytest.mark.parametrize("other", [False, True])
def test_build_does_not_wait_for_another_streams_query(dev, other):
    """A build and a refit on one stream after a BVH that a query on another stream still reads
    was destroyed (and, other, after it a BVH that only this stream has used): they take other
    memory and return while that query is still to run."""
    w = W.cpq_small(n_queries=4096)
    V, F, Q = _t(w["verts"], dev), _t(w["tris"], dev), _t(w["queries"], dev)
    V2, V3 = V * 2.0, V * 3.0
    ctx = gpurt.Context(0)
    busy, side = _two_queues(dev)
    done = torch.cuda.Event()
    with torch.cuda.stream(side):
        own, bvh = gpurt.Bvh(ctx, V, F), gpurt.Bvh(ctx, V, F)
        own.closest_point(Q)
        want = bvh.closest_point(Q)
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        bvh.closest_point(Q)
        _sleep(busy, 0.5)
        got = bvh.closest_point(Q)
        done.record(busy)
    bvh.close()
    if other:
        own.close()
    with torch.cuda.stream(side):
        after = gpurt.Bvh(ctx, V2, F)
        after.refit(V3)
    assert not done.query(), "the build waited for the other stream"
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    for b in (after, own):
        b.close()
    ctx.close()


def test_rebuilding_in_a_loop_takes_no_new_memory(dev):
    """Build, query and destroy on one stream, without waiting: the next build takes the memory
    of the last, so the device's free memory stays as it is."""
    V, F = _soup(1_000_000, dev)
    Q = V[:65536].contiguous()
    ctx = gpurt.Context(0)
    out = None
    for k in range(24):
        bvh = gpurt.Bvh(ctx, V, F)
        out = bvh.closest_point(Q, out=out)
        bvh.close()
        if k == 3:
            torch.cuda.synchronize()
            free = torch.cuda.mem_get_info(dev)[0]
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info(dev)[0] > free - (64 << 20)
    ctx.close()


def test_idle_memory_is_given_up_when_memory_is_short(dev):
    """Memory that a context keeps idle is freed for its other allocations: with a gigabyte free
    on the device and several idle, the scratch of a backward call (84 bytes a query, 2.1 GB) and
    then a build are made."""
    V, F = _soup(2_000_000, dev)
    ctx = gpurt.Context(0, vertex_sums="fixed")
    bvh = gpurt.Bvh(ctx, V, F)
    n = 20_000_000
    q = V.repeat(4, 1)[:n].contiguous()
    prim, pt, dist, bary = bvh.closest_point(q)
    g, gv = torch.ones(n, device=dev), torch.zeros_like(V)
    idle = [gpurt.Bvh(ctx, V, F) for _ in range(12)]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free0 = torch.cuda.mem_get_info(dev)[0]
    for b in idle:
        b.close()
    assert torch.cuda.mem_get_info(dev)[0] < free0 + (1 << 30)  # (kept)
    hog = torch.empty(torch.cuda.mem_get_info(dev)[0] - (1 << 30), dtype=torch.uint8, device=dev)
    bvh.closest_point_bwd(q, prim, bary, pt, dist, g, None, gv)
    other = gpurt.Bvh(ctx, V, F)
    torch.cuda.synchronize()
    assert torch.isfinite(gv).all()
    p2 = other.closest_point(q[:4096])[0]
    assert torch.equal(p2, prim[:4096])
    del hog, q, pt, bary, g, gv
    other.close()
    bvh.close()
    ctx.close()
    torch.cuda.empty_cache()


def test_default_vertex_sums_without_memory_for_scratch(dev):
    """The default mode falls back to atomics, which need no scratch, where the fixed order's (84
    bytes a query) cannot be had: within 2 c^2 2^-24 for vertices of up to c terms of at most 1."""
    V, F = _soup(2_000_000, dev)
    n = 20_000_000
    q = (V.repeat(4, 1)[:n] + 0.002).contiguous()
    g, got = torch.ones(n, device=dev), []
    for mode in ("fixed", "auto"):
        ctx = gpurt.Context(0, vertex_sums=mode)
        bvh = gpurt.Bvh(ctx, V, F)
        prim, pt, dist, bary = bvh.closest_point(q)
        gv = torch.zeros_like(V)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        hog = None
        if mode == "auto":
            hog = torch.empty(torch.cuda.mem_get_info(dev)[0] - (1 << 29), dtype=torch.uint8, device=dev)
        bvh.closest_point_bwd(q, prim, bary, pt, dist, g, None, gv)
        torch.cuda.synchronize()
        del hog
        got.append(gv)
        bvh.close()
        ctx.close()
    c = float(torch.bincount(F.long()[prim.long()].reshape(-1)).max())
    assert float(got[0].abs().max()) > 0
    assert float((got[0] - got[1]).abs().max()) <= 2.0 * c * c * 2.0**-24
    del q, g, pt, bary, got
    torch.cuda.empty_cache()


def test_build_on_a_captured_stream_is_refused(dev):
    """A build on a stream that is being captured is refused (it reads a report back) and takes no
    memory of the graph into the context's pool: the capture is whole, and later builds on the
    stream work."""
    w = W.cpq_small(n_queries=64)
    V, F, Q = _t(w["verts"], dev), _t(w["tris"], dev), _t(w["queries"], dev)
    ep, _, ed, _ = O.cpq_brute_f32(w["verts"], w["tris"], w["queries"])
    ctx = gpurt.Context(0)
    x = torch.arange(1024, dtype=torch.float32, device=dev)
    y = torch.zeros_like(x)
    cap = torch.cuda.Stream(dev)
    for warm in (False, True):  # with nothing in the pool, and with blocks that would fit
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=cap):
            torch.add(x, 1.0, out=y)
            with pytest.raises(gpurt.GpurtError):
                gpurt.Bvh(ctx, V, F)
            torch.mul(y, 2.0, out=y)
        for _ in range(2):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, (x + 1.0) * 2.0)
        with torch.cuda.stream(cap):
            bvh = gpurt.Bvh(ctx, V, F)
            prim, _, dist, _ = bvh.closest_point(Q)
        torch.cuda.synchronize()
        assert np.array_equal(prim.cpu().numpy(), ep) and np.array_equal(dist.cpu().numpy(), ed)
        bvh.close()
    ctx.close()
