"""The work that is timed: what a program does with this package, call by call.

A case is a dict of plain values.  Its "kind" names the call:

  points     closest points of a query set on one mesh            Bvh.closest_point
  rays       one closest-hit and one any-hit pass of a ray set    Bvh.trace_closest, Bvh.trace_any
  instanced  the same through a two-level structure               Tlas.trace_closest, Tlas.trace_any
  step       an optimisation step: distances and hit distances    closest_point_distance, ray_hit_t
             with the gradients of queries, rays and vertices     and torch.autograd
  rebuild    a mesh that changed: build its BVH, trace rays       Bvh(...), Bvh.trace_closest
  refit      vertices that moved: refit, closest points           Bvh.refit, Bvh.closest_point
  batch      many uneven meshes rebuilt and queried, forward      Batch.run, Batch.backward
             and backward
  render     one frame of the path tracer                         tracer.Scene.render

Meshes are noise-displaced spheres and terrains with spheres over them, as in the
package's own workloads, made on the GPU from the seed.  Spheres are cube spheres of
12 g^2 triangles, so that every size can be had.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-rt_amd"))

import gpurt  # noqa: E402
from gpurt import tracer, workloads  # noqa: E402

DEV = torch.device("cuda", 0)
F64 = torch.float64
EXACT_PAIRS = 3e9  # query-triangle pairs that a 64-bit brute force goes through in seconds


def listed():
    return [
        # an interactive probe: a handful of points against a small mesh, all latency
        {"name": "points_probe", "kind": "points", "g": 10, "queries": 100, "mix": "uniform", "treelet": 0},
        # distances around a small object (a collision shape), queries all over its box
        {"name": "points_small_mesh", "kind": "points", "g": 21, "queries": 65536, "mix": "uniform", "treelet": 0},
        # a scan against a dense model: most points near the surface, some far outside or inside
        {"name": "points_dense_mesh", "kind": "points", "g": 661, "queries": 1048576, "mix": "mixed", "treelet": 7},
        # incoherent rays of a renderer or a visibility query through a static scene
        {"name": "rays_scene", "kind": "rays", "grid": 708, "spheres": 64, "g": 41, "rays": 1048576, "treelet": 7},
        # the same scene laid out as instances, an odd number of rays (one bounce of a frame)
        {"name": "instanced_scene", "kind": "instanced", "grid": 708, "spheres": 64, "g": 41, "rays": 500009},
        # one step of fitting a small mesh to points and depths
        {"name": "step_small", "kind": "step", "g": 41, "queries": 30011, "rays": 10007, "treelet": 0, "stride": 3},
        # one step of fitting a 1.3 M triangle mesh
        {"name": "step_large", "kind": "step", "g": 331, "queries": 1048576, "rays": 262144, "treelet": 7, "stride": 3},
        # a small deforming object rebuilt every frame, in the 48-byte vertex record
        {"name": "rebuild_small", "kind": "rebuild", "grid": 0, "spheres": 1, "g": 21, "rays": 4096, "treelet": 0,
         "stride": 12},
        # a scene loaded: the build with the best tree, and its first rays
        {"name": "rebuild_scene", "kind": "rebuild", "grid": 708, "spheres": 64, "g": 41, "rays": 262144, "treelet": 7,
         "stride": 3},
        # simulation: the vertices moved, the tree is refitted, contact points are looked up
        {"name": "refit_contacts", "kind": "refit", "g": 145, "queries": 65536, "treelet": 7, "stride": 3},
        # a training batch of 256 uneven meshes, forward and backward
        {"name": "batch_256", "kind": "batch", "meshes": 256, "tri_hi": 131072, "q_hi": 65536, "data": 6},
        # one progressive frame with multiple importance sampling
        {"name": "render_mis", "kind": "render", "width": 640, "height": 360, "samples": 4, "depth": 8,
         "integrator": "mis", "brdf": "blinn-phong", "sphere_level": 5},
    ]


def draw(rng):
    def size(lo, hi):  # spread over the logarithm, odd as often as not
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["points", "points", "rays", "instanced", "step", "step", "rebuild", "rebuild", "refit", "batch",
                       "render"])
    if kind == "points":
        return {"kind": kind, "g": size(4, 600), "queries": size(16, 900000),
                "mix": rng.choice(["uniform", "near", "mixed"]) if rng.random() < 0.5 else "mixed",
                "treelet": rng.choice([0, 7])} if rng.random() < 0.6 else \
            {"kind": kind, "g": size(4, 128), "queries": size(16, 100000), "mix": "uniform",
             "treelet": rng.choice([0, 7])}
    if kind == "rays":
        return {"kind": kind, "grid": size(16, 700), "spheres": rng.randint(0, 64), "g": size(4, 41),
                "rays": size(100, 1000000), "treelet": rng.choice([0, 5, 7])}
    if kind == "instanced":
        return {"kind": kind, "grid": size(16, 700), "spheres": rng.randint(1, 64), "g": size(4, 41),
                "rays": size(100, 500000)}
    if kind == "step":
        return {"kind": kind, "g": size(8, 331), "queries": size(256, 1000000), "rays": size(64, 250000),
                "treelet": rng.choice([0, 7]), "stride": rng.choice([3, 3, 4, 12])}
    if kind == "rebuild":
        return {"kind": kind, "grid": rng.choice([0, size(8, 700)]), "spheres": rng.randint(1, 64), "g": size(2, 41),
                "rays": size(64, 250000), "treelet": rng.choice([0, 0, 5, 6, 7]), "stride": rng.choice([3, 3, 4, 12])}
    if kind == "refit":
        return {"kind": kind, "g": size(8, 300), "queries": size(100, 100000), "treelet": rng.choice([0, 7]),
                "stride": rng.choice([3, 3, 4, 12])}
    if kind == "batch":
        return {"kind": kind, "meshes": size(2, 200), "tri_hi": size(4096, 131072), "q_hi": size(1024, 65536),
                "data": rng.randint(0, 10 ** 6)}
    return {"kind": "render", "width": size(64, 640), "height": size(64, 360), "samples": rng.randint(1, 4),
            "depth": rng.randint(2, 8), "integrator": rng.choice(["direct", "mats", "mis"]),
            "brdf": rng.choice(["blinn-phong", "ggx"]), "sphere_level": rng.randint(2, 5)}


# ---- meshes and queries, on the GPU ----------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rand(gen, *shape):
    return torch.rand(*shape, generator=gen, device=DEV, dtype=F64)


def _dirs(gen, n):
    d = torch.randn(n, 3, generator=gen, device=DEV, dtype=F64)
    return d / d.norm(dim=1, keepdim=True)


def _waves(gen, p, lo, hi, count=24):
    """Smooth noise of about unit range: waves of random direction with frequencies lo..hi,
    amplitude falling with the frequency."""
    f = torch.exp(_rand(gen, count) * math.log(hi / lo)) * lo
    k = _dirs(gen, count) * f[:, None]
    a = 1.0 / f
    return torch.sin(p @ k.T + 2 * math.pi * _rand(gen, count)) @ (a / a.norm())


def _sphere_grid(g):
    """Unit cube sphere: 6 (g + 1)^2 vertices, 12 g^2 triangles."""
    u = torch.tan(torch.linspace(-math.pi / 4, math.pi / 4, g + 1, device=DEV, dtype=F64))
    b, a = torch.meshgrid(u, u, indexing="ij")
    one = torch.ones_like(a)
    faces = [torch.stack(c, -1).reshape(-1, 3) for c in ((one, a, b), (-one, b, a), (b, one, a), (a, -one, b),
                                                        (a, b, one), (b, a, -one))]
    v = torch.cat(faces)
    v = v / v.norm(dim=1, keepdim=True)
    return v, torch.cat([_grid_tris(g + 1, g + 1) + k * (g + 1) ** 2 for k in range(6)])


def _grid_tris(rows, cols):
    i = torch.arange(rows - 1, device=DEV)[:, None] * cols + torch.arange(cols - 1, device=DEV)[None, :]
    i = i.reshape(-1)
    return torch.stack([torch.stack([i, i + cols, i + 1], 1), torch.stack([i + 1, i + cols, i + cols + 1], 1)],
                       1).reshape(-1, 3)


def _blob(gen, g, amp=0.05):
    v, f = _sphere_grid(g)
    return v * (1.0 + amp * _waves(gen, v, 2.0, 16.0))[:, None], f


def _terrain(gen, grid, extent=50.0, height=2.5):
    x = torch.linspace(-extent, extent, grid, device=DEV, dtype=F64)
    z, x = torch.meshgrid(x, x, indexing="ij")
    p = torch.stack([x.reshape(-1), torch.zeros(grid * grid, device=DEV, dtype=F64), z.reshape(-1)], 1)
    y = height * _waves(gen, p / 20.0, 1.0, 32.0, 32)
    return torch.stack([p[:, 0], y, p[:, 2]], 1), _grid_tris(grid, grid)


def _placements(gen, n, lo, hi):
    c = torch.stack([_rand(gen, n) * 90 - 45, _rand(gen, n) * (hi + 8 - lo) + lo, _rand(gen, n) * 90 - 45], 1)
    return c, _rand(gen, n) * 2.5 + 0.5


def _scene(gen, grid, spheres, g):
    """Terrain with spheres over it as one mesh (grid 0: the spheres alone)."""
    vs, fs, off, lo, hi = [], [], 0, -3.0, 3.0
    if grid:
        v, f = _terrain(gen, grid)
        vs, fs, off = [v], [f], v.shape[0]
        lo, hi = float(v[:, 1].min()), float(v[:, 1].max())
    if spheres:
        sv, sf = _blob(gen, g)
        c, r = _placements(gen, spheres, lo, hi)
        vs.append((sv[None] * r[:, None, None] + c[:, None]).reshape(-1, 3))
        fs.append((sf[None] + off + torch.arange(spheres, device=DEV)[:, None, None] * sv.shape[0]).reshape(-1, 3))
    return torch.cat(vs), torch.cat(fs)


def _verts(v, stride=3):
    out = torch.zeros(v.shape[0], stride, device=DEV, dtype=torch.float32)
    out[:, :3] = v
    return out


def _near(gen, v, f, n, sigma=0.005):
    t = f[torch.randint(0, f.shape[0], (n,), generator=gen, device=DEV)]
    a, b, c = v[t[:, 0]], v[t[:, 1]], v[t[:, 2]]
    s, u = _rand(gen, n, 1).sqrt(), _rand(gen, n, 1)
    nrm = torch.linalg.cross(b - a, c - a)
    nrm = nrm / nrm.norm(dim=1, keepdim=True).clamp_min(1e-300)
    return (1 - s) * a + s * (1 - u) * b + s * u * c + nrm * torch.randn(n, 1, generator=gen, device=DEV, dtype=F64) * sigma


def _queries(gen, v, f, n, mix, box=2.0):
    k = {"near": n, "uniform": 0, "mixed": int(0.8 * n)}[mix]
    q = torch.cat([_near(gen, v, f, k), (_rand(gen, n - k, 3) * 2 - 1) * (1.5 if mix == "uniform" else box)])
    return q[torch.randperm(n, generator=gen, device=DEV)].float().contiguous()


def _rays(o, d, tmin=1e-5, tmax=1e7):
    return gpurt.make_rays(o.float(), d.float(), tmin, tmax)


def _box_rays(gen, lo, hi, n):
    """Incoherent rays in a box, for closest hit and (bounded) for any hit."""
    o, d = lo + (hi - lo) * _rand(gen, n, 3), _dirs(gen, n)
    return _rays(o, d), _rays(o, d, 1e-5, (_rand(gen, n) * 49 + 1).float())


def _inward_rays(gen, n, centre=0.0, radius=3.0, target=0.5):
    o = _dirs(gen, n) * radius
    d = _dirs(gen, n) * target * _rand(gen, n, 1) - o
    return centre + o, d / d.norm(dim=1, keepdim=True)


def _batch_sizes(case):
    gen = torch.Generator().manual_seed(case["data"])
    m = case["meshes"]
    u, w = torch.rand(m, generator=gen, dtype=F64), torch.rand(m, generator=gen, dtype=F64)
    tris = torch.exp(math.log(1024) + u * math.log(case["tri_hi"] / 1024)).tolist()
    n = torch.exp(math.log(256) + w * math.log(case["q_hi"] / 256)).long().tolist()
    return [(max(2, round(math.sqrt(t / 12.0 if k % 2 == 0 else t / 2.0))), n[k]) for k, t in enumerate(tris)]


def _batch_mesh(gen, k, g, n):
    if k % 2 == 0:
        v, f = _blob(gen, g)
    else:
        v, f = _terrain(gen, g + 1)
        v = v / 50.0
    v32 = _verts(v)
    lo, hi = v.min(0).values, v.max(0).values
    mid, half = (lo + hi) / 2, (hi - lo) / 2 * 1.2
    k = int(0.8 * n)
    q = torch.cat([_near(gen, v, f, k), mid + (_rand(gen, n - k, 3) * 2 - 1) * half])
    q = q[torch.randperm(n, generator=gen, device=DEV)].float().contiguous()
    o, d = _inward_rays(gen, n, v.mean(0), 1.5 * float(half.norm()), 0.7 * float(half.norm()))
    return {"verts": v32, "tris": f.int().contiguous(), "queries": q, "rays": _rays(o, d)}


# ---- the calls -------------------------------------------------------------------------


def _inputs(case, seed):
    """The tensors of a single-mesh case, from the seed alone."""
    gen, kind, s = _gen(seed), case["kind"], {}
    if kind in ("rays", "rebuild"):
        v, f = _scene(gen, case["grid"], case["spheres"], case["g"])
        s["rays"], s["rays_any"] = _box_rays(gen, v.min(0).values, v.max(0).values, case["rays"])
    else:
        v, f = _blob(gen, case["g"])
        if kind == "refit":
            s["verts0"] = _verts(v, case["stride"])
            v = v * (1.0 + 0.02 * _waves(gen, v, 2.0, 8.0))[:, None]
        mix = case.get("mix", "near")
        s["q"] = _queries(gen, v, f, case["queries"], mix)
        if kind == "step":
            o, d = _inward_rays(gen, case["rays"])
            s["o"], s["d"] = o.float().contiguous(), d.float().contiguous()
            s["g_dist"] = torch.randn(case["queries"], generator=gen, device=DEV)
            s["g_t"] = torch.randn(case["rays"], generator=gen, device=DEV)
    s["verts"], s["tris"] = _verts(v, case.get("stride", 3)), f.int().contiguous()
    return s


def prepare(case, seed):
    ctx, kind = gpurt.default_context(0), case["kind"]
    if kind == "batch":
        gen = _gen(seed)
        meshes = [_batch_mesh(gen, k, g, n) for k, (g, n) in enumerate(_batch_sizes(case))]
        b = gpurt.Batch(ctx, meshes)
        grads = b.enable_backward()
        for g in grads:
            g["g_dist"].normal_(generator=gen)
            g["g_t"].normal_(generator=gen)
        return {"kind": kind, "batch": b}
    if kind == "instanced":
        gen = _gen(seed)
        tv, tf = _terrain(gen, case["grid"])
        sv, sf = _blob(gen, case["g"])
        lo, hi = tv.min(0).values, tv.max(0).values
        c, r = _placements(gen, case["spheres"], float(lo[1]), float(hi[1]))
        rot = torch.linalg.qr(torch.randn(case["spheres"], 3, 3, generator=gen, device=DEV, dtype=F64)).Q
        xf = torch.cat([rot * r[:, None, None], c[:, :, None]], 2).cpu()
        terrain = gpurt.Bvh(ctx, _verts(tv), tf.int().contiguous(), treelet_size=7)
        sphere = gpurt.Bvh(ctx, _verts(sv), sf.int().contiguous(), treelet_size=7)
        t = gpurt.Tlas(ctx, [(terrain, torch.eye(3, 4, dtype=F64))] + [(sphere, m) for m in xf])
        hi = torch.maximum(hi, (c + r[:, None]).max(0).values)
        rays, rays_any = _box_rays(gen, lo, hi, case["rays"])
        return {"kind": kind, "tlas": t, "rays": rays, "rays_any": rays_any}
    if kind == "render":
        w = workloads.tracer_box(case["sphere_level"])
        gen = torch.Generator().manual_seed(seed)
        at = (torch.rand(3, generator=gen, dtype=F64) * 2 - 1).tolist()
        cam = tracer.camera((at[0], at[1], 14.0 + at[2]), w["camera"]["target"], yfov_deg=w["camera"]["yfov_deg"],
                            aspect=case["width"] / case["height"])
        return {"kind": kind, "case": case, "scene": tracer.Scene(ctx, w["objects"]), "camera": cam, "seed": seed}
    s = dict(_inputs(case, seed), kind=kind)
    if kind == "rebuild":
        s["treelet"] = case["treelet"]
        return s
    s["bvh"] = gpurt.Bvh(ctx, s["verts0"] if kind == "refit" else s["verts"], s["tris"], treelet_size=case["treelet"])
    if kind == "step":
        for k in ("q", "o", "d", "verts"):
            s[k].requires_grad_(True)
    return s


def run(s):
    kind = s["kind"]
    if kind == "points":
        return s["bvh"].closest_point(s["q"])
    if kind == "rays":
        return s["bvh"].trace_closest(s["rays"]) + (s["bvh"].trace_any(s["rays_any"]),)
    if kind == "instanced":
        return s["tlas"].trace_closest(s["rays"]) + (s["tlas"].trace_any(s["rays_any"]),)
    if kind == "step":
        dist, prim = gpurt.closest_point_distance(s["bvh"], s["q"], s["verts"])
        t, hit = gpurt.ray_hit_t(s["bvh"], s["o"], s["d"], s["verts"])
        grads = torch.autograd.grad([dist, t], [s["q"], s["o"], s["d"], s["verts"]], [s["g_dist"], s["g_t"]])
        return {"dist": dist, "prim": prim, "t": t, "hit": hit, "grads": grads}
    if kind == "rebuild":
        bvh = gpurt.Bvh(gpurt.default_context(0), s["verts"], s["tris"], treelet_size=s["treelet"])
        out = bvh.trace_closest(s["rays"])
        bvh.close()
        return out
    if kind == "refit":
        s["bvh"].refit(s["verts"])
        return s["bvh"].closest_point(s["q"])
    if kind == "batch":
        out, grads = s["batch"].run(), s["batch"].backward()
        # one tensor per quantity over all meshes, as a loss over the batch reads them
        r = {k: torch.cat([m[k] for m in out]) for k in out[0]}
        return dict(r, **{k: torch.cat([m[k] for m in grads]) for k in ("g_q", "g_origin", "g_dir", "g_verts")})
    c = s["case"]
    return s["scene"].render(c["width"], c["height"], *s["camera"], samples=c["samples"], max_depth=c["depth"],
                             integrator=c["integrator"], brdf=c["brdf"], env_light=0.1, seed=s["seed"])


# ---- what a pass cannot do without -----------------------------------------------------


def _n_tris(case):
    if case["kind"] in ("rays", "rebuild", "instanced"):
        instances = 1 if case["kind"] == "instanced" else case["spheres"]
        return 2 * max(0, case["grid"] - 1) ** 2 + instances * 12 * case["g"] ** 2
    return 12 * case["g"] ** 2


def work(case):
    """Bytes: each triangle's positions once (36 B; 48 B with its indices where it is built
    from), inputs once, outputs once.  Operations: one root-to-leaf descent of a 4-wide
    tree per query (20 per box), one triangle at its end (60)."""
    kind = case["kind"]

    def descents(n, tris):
        return n * (80.0 * math.log(max(tris, 4), 4) + 60.0)

    if kind == "batch":
        b = f = 0.0
        for k, (g, n) in enumerate(_batch_sizes(case)):
            tris, verts = (12 * g * g, 6 * (g + 1) ** 2) if k % 2 == 0 else (2 * g * g, (g + 1) ** 2)
            b += 48.0 * tris + n * (12 + 32 + 32 + 16) + n * (4 + 12) + n * (4 + 24) + 12 * verts
            f += descents(2 * n, tris) + 100.0 * tris
        return {"bytes": b, "flops": f}
    if kind == "render":
        px = case["width"] * case["height"]
        tris = 2 * 20 * 4 ** case["sphere_level"]
        paths = px * case["samples"]
        return {"bytes": 16.0 * px + 144.0 * tris / 2, "flops": descents(2.0 * paths, tris)}
    tris = _n_tris(case)
    if kind == "points":
        n = case["queries"]
        return {"bytes": 36.0 * tris + n * (12 + 32), "flops": descents(n, tris)}
    if kind == "rays" or kind == "instanced":
        n = case["rays"]
        out = 16 + 1 + (4 if kind == "instanced" else 0)
        return {"bytes": 36.0 * tris + n * (64 + out), "flops": descents(2 * n, tris)}
    verts = 6 * (case["g"] + 1) ** 2
    if kind == "step":
        n, m = case["queries"], case["rays"]
        return {"bytes": 36.0 * tris + n * (12 + 4 + 8 + 12) + m * (24 + 4 + 8 + 24) + 4.0 * case["stride"] * verts,
                "flops": descents(n + m, tris) + 150.0 * (n + m)}
    if kind == "rebuild":
        return {"bytes": 48.0 * tris + case["rays"] * 48.0, "flops": 100.0 * tris + descents(case["rays"], tris)}
    return {"bytes": 48.0 * tris + case["queries"] * 44.0, "flops": 50.0 * tris + descents(case["queries"], tris)}


# ---- 64-bit results, by brute force ----------------------------------------------------


def _dot(a, b):
    return (a * b).sum(-1)


def _on_triangle(p, a, b, c):
    """Closest point of each triangle (broadcast against p): squared distance and weights."""
    best = w = None
    corners = (a, b, c)
    for i, j in ((0, 1), (1, 2), (2, 0)):
        e = corners[j] - corners[i]
        s = (_dot(p - corners[i], e) / _dot(e, e).clamp_min(1e-300)).clamp(0.0, 1.0)
        r = p - corners[i] - s[..., None] * e
        d2, ws = _dot(r, r), [torch.zeros_like(s)] * 3
        ws[i], ws[j] = 1 - s, s
        if best is None:
            best, w = d2, ws
        else:
            w = [torch.where(d2 < best, y, x) for x, y in zip(w, ws)]
            best = torch.minimum(best, d2)
    n = torch.linalg.cross(b - a, c - a)
    nn = _dot(n, n).clamp_min(1e-300)
    wb = _dot(torch.linalg.cross(p - a, (c - a).expand(torch.broadcast_shapes(p.shape, a.shape))), n) / nn
    wc = _dot(torch.linalg.cross((b - a).expand(torch.broadcast_shapes(p.shape, a.shape)), p - a), n) / nn
    inside = (wb >= 0) & (wc >= 0) & (wb + wc <= 1)
    h2 = _dot(p - a, n) ** 2 / nn
    face = inside & (h2 <= best)
    w = [torch.where(face, y, x) for x, y in zip(w, (1 - wb - wc, wb, wc))]
    return torch.where(face, h2, best), torch.stack(w, -1)


def _hit(o, d, a, b, c, tmin, tmax):
    """Hit distance (inf: none), u and v of rays and triangles (broadcast)."""
    e1, e2 = b - a, c - a
    shape = torch.broadcast_shapes(o.shape, a.shape)
    p = torch.linalg.cross(d.expand(shape), e2.expand(shape))
    inv = 1.0 / _dot(e1, p)
    s = o - a
    u = _dot(s, p) * inv
    q = torch.linalg.cross(s, e1.expand(shape))
    v = _dot(d, q) * inv
    t = _dot(e2, q) * inv
    ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= tmin) & (t <= tmax)
    return torch.where(ok, t, torch.full_like(t, math.inf)), u, v


def _closest(q, v, f):
    q, tri = q.to(F64), v[:, :3].to(F64)[f.long()]
    a, b, c = tri[:, 0], tri[:, 1], tri[:, 2]
    step = max(1, int(4e6 // f.shape[0]))
    i = torch.cat([_on_triangle(x[:, None], a, b, c)[0].argmin(1) for x in q.split(step)])
    d2, w = _on_triangle(q, a[i], b[i], c[i])
    return i, (w[:, :, None] * tri[i]).sum(1), d2.sqrt(), w


def _first_hits(rays, v, f):
    rays, tri = rays.to(F64), v[:, :3].to(F64)[f.long()]
    a, b, c = tri[:, 0], tri[:, 1], tri[:, 2]
    step = max(1, int(4e6 // f.shape[0]))

    def parts(r):
        return r[..., 0:3], r[..., 4:7], r[..., 3], r[..., 7]

    i = []
    for r in rays.split(step):
        o, d, lo, hi = parts(r[:, None])
        i.append(_hit(o, d, a, b, c, lo, hi)[0].argmin(1))
    i = torch.cat(i)
    o, d, lo, hi = parts(rays)
    t, u, w = _hit(o, d, a[i], b[i], c[i], lo, hi)
    uv = torch.where(torch.isfinite(t)[:, None], torch.stack([u, w], 1), torch.zeros_like(t)[:, None])
    return i, t, uv


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "instanced", "render"):
        return None
    pairs = _n_tris(case) * (case.get("queries", 0) + case.get("rays", 0))
    if pairs > EXACT_PAIRS:
        return None
    s = _inputs(case, seed)
    v, f = s["verts"], s["tris"]
    if kind in ("points", "refit"):
        # (a point over an edge or a corner belongs to several triangles: weights and id are
        # those of the lowest one, the point and the distance are everybody's)
        _, pt, dist, _ = _closest(s["q"], v, f)
        return None, pt, dist, None
    if kind in ("rays", "rebuild"):
        _, t, uv = _first_hits(s["rays"], v, f)
        return (None, t, uv, None)[:4 if kind == "rays" else 3]
    # distances: d = |q - p|, dd/dq = (q - p) / d, dd/dv_j = -w_j dd/dq; hit distances:
    # dt/do = -n / (n . d), dt/dd = t dt/do, dt/dv_j = -w_j dt/do
    f = f.long()
    i, pt, dist, w = _closest(s["q"], v, f)
    g = (s["q"].to(F64) - pt) / dist[:, None].clamp_min(1e-300) * s["g_dist"].to(F64)[:, None]
    gv = torch.zeros(v.shape, device=DEV, dtype=F64)
    for j in range(3):
        gv[:, :3].index_add_(0, f[i, j], -w[:, j:j + 1] * g)
    h, t, uv = _first_hits(_rays(s["o"], s["d"]), v, f)
    tri, live = v[:, :3].to(F64)[f[h]], torch.isfinite(t)
    n = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    go = -n / _dot(n, s["d"].to(F64))[:, None] * s["g_t"].to(F64)[:, None]
    go = torch.where(live[:, None], go, torch.zeros_like(go))
    gd = go * torch.where(live, t, torch.zeros_like(t))[:, None]
    wr = torch.stack([1 - uv[:, 0] - uv[:, 1], uv[:, 0], uv[:, 1]], 1)
    for j in range(3):
        gv[:, :3].index_add_(0, f[h, j], -wr[:, j:j + 1] * go)
    return {"dist": dist, "prim": None, "t": t, "hit": None, "grads": (g, go, gd, gv)}
