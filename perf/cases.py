"""Performance cases of the ray-space accelerators, through the Python binding's public calls.

One pass of a case is what a renderer or a render service has the library do once:
  direct    closest hits of a camera image, point-light shadow rays from them, their occlusion
            (the directlighting integrator's step over one image or one task of a frame)
  path      the same followed by diffuse bounces, a shadow pass at every depth (path integrator)
  segments  occlusion of unstructured segments (visibility queries, many-light shadow rays)
  batch     closest hits and occlusion of many scenes in one batched launch (graph replay)
  serve     requests handed to the serving loop together and waited for
Scenes and cameras are those of pbrt-v2_amd/scenes.py; every array depends on the seed.
"""
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent

# camera position, vertical field of view and point light of each scene family
VIEWS = {
    "random": ((0.0, 0.0, -3.0), 60.0, (2.0, 2.0, -2.0)),
    "torus": ((0.0, 0.0, -3.0), 60.0, (2.0, 2.0, -2.0)),
    "clusters": ((0.0, 0.0, -12.0), 50.0, (2.0, 2.0, -2.0)),
    "room": ((0.0, 0.0, -9.0), 50.0, (1.0, 2.5, -8.0)),
}
TORUS_TRIS = 24778
DEVICE = "cuda"


def _package():
    """The library's Python binding and its scene generators (the directory is not an identifier)."""
    for name, path, search in (("pbrt_v2_amd", ROOT / "pbrt-v2_amd" / "__init__.py",
                                [str(ROOT / "pbrt-v2_amd")]),
                               ("pbrt_v2_amd.scenes", ROOT / "pbrt-v2_amd" / "scenes.py", None)):
        if name not in sys.modules:
            spec = importlib.util.spec_from_file_location(name, path,
                                                          submodule_search_locations=search)
            mod = importlib.util.module_from_spec(spec)
            sys.modules[name] = mod
            spec.loader.exec_module(mod)
    return sys.modules["pbrt_v2_amd"], sys.modules["pbrt_v2_amd.scenes"]


rt, scenes = _package()
_context = None


def _ctx():
    global _context
    if _context is None:
        _context = rt.Context(0)
    return _context


# ---------------------------------------------------------------------------------------
# the cases

def _case(name, kind, **kw):
    c = dict(name=name, kind=kind, accel="rayhierarchy", node="box_dir", scene="torus",
             ntri=TORUS_TRIS, width=256, height=256, spp=1, chunk_x=4, chunk_y=4, levels=3,
             shading=False, keep=False, depth=0, count=1)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call a program makes: a preview image of a small scene; launches and
        # latency decide it
        _case("preview_64", "direct", scene="random", ntri=1024, width=64, height=64),
        # the naive accelerator's configuration: 1,024 random triangles, 128 x 128
        _case("naive_128", "direct", accel="naive", scene="random", ntri=1024, width=128,
              height=128),
        # the rayhierarchy workload: torus, 512 x 512, directlighting, buffers kept by the
        # renderer from frame to frame
        _case("torus_512", "direct", width=512, height=512, keep=True),
        # interval-arithmetic nodes, an image no tile divides, and the shading record
        _case("torus_ia_odd", "direct", node="ia", width=333, height=251, shading=True),
        # the accelerator line of the reference's scene files (100 x 4 leaves, ia): blocks of
        # 6,400 rays
        _case("scene_file_blocks", "direct", node="ia", scene="clusters", ntri=20000, width=400,
              height=300, chunk_x=100),
        # node "box_uv" over a medium scene
        _case("clusters_uv", "direct", node="box_uv", scene="clusters", ntri=12000, width=240,
              height=180),
        # ray-bvh: one 256 x 256 x 4 spp task of the room frame, directlighting
        _case("room_task", "direct", accel="ray-bvh", scene="room", ntri=80012, width=256,
              height=256, spp=4, keep=True),
        # the same task through the path integrator to depth 3
        _case("room_path3", "path", accel="ray-bvh", scene="room", ntri=80012, width=256,
              height=256, spp=4, depth=3),
        # a large scene at full resolution, directlighting: shadow rays from scattered points
        _case("clusters_1024", "direct", scene="clusters", ntri=200000, width=1024, height=1024,
              keep=True),
        # a million unstructured visibility segments against the same scene
        _case("segments_1m", "segments", scene="clusters", ntri=200000, width=256, height=4096),
        # twelve scenes of uneven size in one batched launch
        _case("batch_12", "batch", scene="clusters", ntri=100000, width=512, height=512, count=12),
        # the serving loop with eight requests of mixed sizes at once
        _case("serve_8", "serve", scene="clusters", ntri=60000, width=320, height=320, count=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["direct", "direct", "direct", "path", "segments", "batch", "serve"])
    if kind == "batch":
        return _drawn(kind, scene="clusters", ntri=_log_int(rng, 5000, 100000),
                      width=_log_int(rng, 96, 512), height=_log_int(rng, 96, 512),
                      count=rng.randint(2, 12))
    if kind == "serve":
        return _drawn(kind, scene="clusters", ntri=_log_int(rng, 5000, 60000),
                      width=_log_int(rng, 64, 320), height=_log_int(rng, 64, 320),
                      count=rng.randint(1, 8))
    if kind == "segments":
        return _drawn(kind, accel=rng.choice(["rayhierarchy", "ray-bvh"]), scene="clusters",
                      ntri=_log_int(rng, 1000, 200000), width=rng.choice([64, 100, 256, 300]),
                      height=_log_int(rng, 16, 3400))
    if kind == "path":
        return _drawn(kind, accel=rng.choice(["rayhierarchy", "ray-bvh"]), scene="room",
                      ntri=12 + 200 * _log_int(rng, 20, 400), width=_log_int(rng, 64, 256),
                      height=_log_int(rng, 64, 256), spp=rng.choice([1, 2, 4]),
                      depth=rng.randint(1, 3))
    accel = rng.choice(["naive", "rayhierarchy", "rayhierarchy", "rayhierarchy", "ray-bvh",
                        "ray-bvh"])
    if accel == "naive":
        return _drawn(kind, accel=accel, scene="random", ntri=_log_int(rng, 64, 4096),
                      width=_log_int(rng, 32, 256), height=_log_int(rng, 32, 256),
                      shading=rng.random() < 0.3)
    node = rng.choice(["box_dir", "box_dir", "box_dir", "ia", "box_uv"])
    scene = rng.choice(["random", "torus", "clusters", "room"])
    small = node != "box_dir"  # ia and box_uv keep far more of a scene per tile
    ntri = {"random": _log_int(rng, 200, 20000), "torus": TORUS_TRIS,
            "clusters": _log_int(rng, 1000, 12000 if small else 200000),
            "room": 12 + 200 * _log_int(rng, 5, 50 if small else 400)}[scene]
    side = 224 if small else 700
    cx, cy, levels = rng.choice([(4, 4, 3), (4, 4, 3), (4, 4, 2), (2, 4, 4), (8, 4, 3), (100, 4, 3)])
    return _drawn(kind, accel=accel, node=node, scene=scene, ntri=ntri,
                  width=_log_int(rng, 40, side), height=_log_int(rng, 40, side), chunk_x=cx,
                  chunk_y=cy, levels=levels, shading=rng.random() < 0.3, keep=rng.random() < 0.5)


def _drawn(kind, **kw):
    c = _case("", kind, **kw)
    del c["name"]
    return c


# ---------------------------------------------------------------------------------------
# inputs

def _triangles(c, seed, ntri=None):
    ntri = c["ntri"] if ntri is None else ntri
    if c["scene"] == "random":
        return scenes.random_triangles(ntri, seed=seed)
    if c["scene"] == "torus":
        return scenes.torus_scene(seed=seed)
    if c["scene"] == "room":
        return scenes.room_scene(seed=seed, nclusters=max(1, (ntri - 12) // 200))
    return scenes.cluster_scene(ntri, seed=seed)


def _origin(c, seed):
    o = np.array(VIEWS[c["scene"]][0]) + np.random.default_rng(seed).uniform(-0.05, 0.05, 3)
    return tuple(float(x) for x in o)


def _camera(c, seed, width=None, height=None):
    return scenes.pinhole_rays(width or c["width"], height or c["height"], origin=_origin(c, seed),
                               fov_deg=VIEWS[c["scene"]][1], spp=c["spp"], seed=seed)


def _desc(c):
    kw = dict(node=c["node"], chunk_x=c["chunk_x"], chunk_y=c["chunk_y"], height=c["levels"])
    return rt.default_desc(c["accel"], **({} if c["accel"] == "naive" else kw))


def _batch_sizes(c):
    """Triangle and image sizes of a batch's scenes: log-uniform up to the case's own, the first
    one at the full size."""
    g = np.random.default_rng(c["count"])
    out = []
    for i in range(c["count"]):
        f = (1.0, 1.0, 1.0) if i == 0 else np.exp(g.uniform(np.log([0.02, 0.2, 0.2]), 0.0))
        out.append((max(200, int(c["ntri"] * f[0])), max(16, int(c["width"] * f[1])),
                    max(16, int(c["height"] * f[2]))))
    return out


def _serve_sizes(c):
    """Image sizes of the requests: a fixed mix down to a quarter of the case's side."""
    return [(max(16, c["width"] * f // 4), max(16, c["height"] * f // 4))
            for f in (4, 1, 2, 3, 1, 4, 2, 3)[:c["count"]]]


class _State:
    """What a program keeps between passes; closes the library's handles with itself."""

    def __init__(self, **kw):
        self.handles = []
        self.__dict__.update(kw)

    def own(self, handle):
        self.handles.append(handle)
        return handle

    def __del__(self):
        for h in reversed(self.handles):
            h.close()


def _empty_rays(n, width, height):
    f = [torch.empty(n, dtype=torch.float32, device=DEVICE) for _ in range(8)]
    return rt.DeviceRays(*f, torch.empty(n, dtype=torch.uint8, device=DEVICE), width, height)


def prepare(case, seed):
    c = case
    s = _State(case=c)
    if c["kind"] == "batch":
        s.stream = torch.cuda.Stream()
        s.batch = rt.Batch(_ctx())
        s.out = []
        for i, (ntri, w, h) in enumerate(_batch_sizes(c)):
            sc = s.own(rt.Scene(_ctx(), _triangles(c, seed * 64 + i, ntri), desc=_desc(c)))
            cam = rt.DeviceRays.from_numpy(_camera(c, seed * 64 + i, w, h))
            seg = rt.DeviceRays.from_numpy(scenes.random_rays(
                64 * max(1, w * h // 64), seed=seed * 64 + i, width=64))
            hits = s.batch.add_closest(sc, cam)
            s.out.append(dict(id=hits.id, t=hits.t, u=hits.u, v=hits.v,
                              occluded=s.batch.add_occluded(sc, seg)))
        s.own(s.batch)
        s.batch.set_param(rt.RT_PARAM_GRAPH, 1)
        return s
    if c["kind"] == "serve":
        list_ = [s.own(rt.Scene(_ctx(), _triangles(c, seed * 64 + i, max(1000, c["ntri"] >> i)),
                                desc=_desc(c))) for i in range(4)]
        s.server = s.own(rt.Server(_ctx(), list_, mem_budget=1 << 30))
        s.requests = [dict(scene=i % 4, width=w, height=h, origin=_origin(c, seed * 64 + i),
                           fov_deg=VIEWS[c["scene"]][1], light=VIEWS[c["scene"]][2])
                      for i, (w, h) in enumerate(_serve_sizes(c))]
        return s
    s.scene = s.own(rt.Scene(_ctx(), _triangles(c, seed), desc=_desc(c)))
    s.light = VIEWS[c["scene"]][2]
    s.hits = s.shadow = s.occluded = None
    if c["kind"] == "segments":
        s.rays = rt.DeviceRays.from_numpy(scenes.random_rays(c["width"] * c["height"], seed=seed,
                                                             width=c["width"]))
        return s
    s.rays = rt.DeviceRays.from_numpy(_camera(c, seed))
    if c["keep"]:
        n = s.rays.count
        s.hits = rt.DeviceHits.empty(n, shading=c["shading"])
        s.shadow = _empty_rays(n, s.rays.width, s.rays.height)
        s.occluded = torch.empty(n, dtype=torch.uint8, device=DEVICE)
    return s


# ---------------------------------------------------------------------------------------
# one pass

def _record(h):
    out = dict(id=h.id, t=h.t, u=h.u, v=h.v)
    if h.dpdu is not None:
        out.update(dpdu=h.dpdu, dpdv=h.dpdv)
    return out


def run(state):
    s, c = state, state.case
    if c["kind"] == "batch":
        s.batch.run(stream=s.stream)
        return s.out
    if c["kind"] == "serve":
        tickets = [s.server.submit(outputs=True, **q) for q in s.requests]
        done = [s.server.wait(t) for t in tickets]
        return [dict(id=d["id"], t=d["t"], occluded=d["occ"]) for d in done]
    if c["kind"] == "segments":
        return dict(occluded=s.scene.trace_occluded(s.rays))
    hits = s.scene.trace_closest(s.rays, rt.RT_CLOSEST_PRIMARY, hits=s.hits, shading=c["shading"])
    shadow = rt.make_shadow_rays(s.rays, hits, s.light, out=s.shadow)
    out = [dict(_record(hits), occluded=s.scene.trace_occluded(shadow, out=s.occluded))]
    rays = s.rays
    for depth in range(c["depth"]):
        rays = rt.make_bounce_rays(s.scene, rays, hits, seed=7, depth=depth)
        hits = s.scene.trace_closest(rays, rt.RT_CLOSEST_SECONDARY)
        shadow = rt.make_shadow_rays(rays, hits, s.light)
        out.append(dict(_record(hits), occluded=s.scene.trace_occluded(shadow)))
    return out


# ---------------------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    """Bytes: each scene and each given ray read once (36 B per triangle; 32 B per ray, 33 with
    validity), each result written once (16 B per closest hit, 40 with the shading record, 1 B
    per flag).  Operations: 45 per leaf test, one test per ray (naive: every ray tests every
    triangle, which is what that accelerator is)."""
    c = case
    if c["kind"] == "batch":
        sizes = _batch_sizes(c)
        rays = sum(w * h for _, w, h in sizes)
        return dict(bytes=36 * sum(t for t, _, _ in sizes) + rays * (32 + 16 + 33 + 1),
                    flops=90 * rays)
    if c["kind"] == "serve":
        rays = sum(w * h for w, h in _serve_sizes(c))
        return dict(bytes=36 * sum(max(1000, c["ntri"] >> i) for i in range(min(4, c["count"])))
                    + rays * (8 + 1), flops=90 * rays)
    n = c["width"] * c["height"] * c["spp"]
    if c["kind"] == "segments":
        return dict(bytes=36 * c["ntri"] + n * (33 + 1), flops=45 * n)
    per_hit = 40 if c["shading"] else 16
    tests = 2 * n * (1 + c["depth"]) * (c["ntri"] if c["accel"] == "naive" else 1)
    return dict(bytes=36 * c["ntri"] + n * (32 + (per_hit + 1) * (1 + c["depth"])),
                flops=45 * tests)


# ---------------------------------------------------------------------------------------
# the camera pass in 64 bits

def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _cross(a, b):
    return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])


def exact(case, seed):
    """The camera rays' hit records by brute force in 64 bits: for the naive accelerator (every
    triangle, its thresholds) and for rayhierarchy with interval nodes (a conservative cull, so
    every triangle passing the strict test counts).  With box_dir and box_uv nodes, 32-bit cull
    predicates decide which triangles count, and bounces follow 32-bit random directions: no
    such value there, and none for ids and flags, which are whole numbers."""
    c = case
    naive = c["accel"] == "naive"
    if c["kind"] != "direct" or not (naive or (c["node"] == "ia" and c["accel"] == "rayhierarchy")):
        return None
    if c["width"] * c["height"] * c["spp"] * c["ntri"] > 4e9:
        return None
    f64 = dict(dtype=torch.float64, device=DEVICE)
    v = torch.as_tensor(np.asarray(_triangles(c, seed), np.float32).reshape(-1, 9)).to(**f64)
    r = _camera(c, seed)
    rays = [torch.as_tensor(np.ascontiguousarray(r[k])).to(**f64)
            for k in ("ox", "oy", "oz", "dx", "dy", "dz")]
    v1, v2, v3 = (tuple(v[:, 3 * k + a][None] for a in range(3)) for k in range(3))
    e1 = tuple(b - a for a, b in zip(v1, v2))
    e2 = tuple(b - a for a, b in zip(v1, v3))
    n = rays[0].numel()
    t = torch.full((n,), math.inf, **f64)
    u, w = torch.zeros(n, **f64), torch.zeros(n, **f64)
    tri = torch.full((n,), -1, dtype=torch.int64, device=DEVICE)
    step = max(1, int(2e7) // v.shape[0])
    for i in range(0, n, step):
        o = tuple(x[i:i + step, None] for x in rays[:3])
        d = tuple(x[i:i + step, None] for x in rays[3:])
        s1 = _cross(d, e2)
        det = _dot(s1, e1)
        ov = tuple(a - b for a, b in zip(o, v1))
        b1 = _dot(ov, s1) / det
        s2 = _cross(ov, e1)
        b2 = _dot(d, s2) / det
        tt = _dot(e2, s2) / det
        if naive:
            eps = 0.002
            ok = (det.abs() >= eps) & (b1 >= -1e-3 - eps) & (b1 <= 1 + 1e-3 + eps) \
                & (b2 >= -1e-3 - eps) & (b1 + b2 <= 1 + 1e-3 + eps) & (tt >= 0)
        else:
            ok = (b1 > 0) & (b1 < 1) & (b2 > 0) & (b1 + b2 < 1) & (tt > 0)
        best, at = torch.where(ok, tt, math.inf).min(dim=1)
        hit = best < math.inf
        t[i:i + step] = best
        pick = lambda x: torch.where(hit, x.gather(1, at[:, None])[:, 0], 0.0)  # noqa: E731
        # default texture coordinates (0,0), (1,0), (1,1)
        u[i:i + step], w[i:i + step] = pick(b1) + pick(b2), pick(b2)
        tri[i:i + step] = torch.where(hit, at, -1)
    out = dict(id=None, t=t, u=u, v=w, occluded=None)
    if c["shading"]:
        hit = (tri >= 0)[:, None]
        p = v[tri.clamp(min=0)]
        out["dpdu"] = torch.where(hit, p[:, 3:6] - p[:, 0:3], 0.0).reshape(-1)
        out["dpdv"] = torch.where(hit, p[:, 6:9] - p[:, 3:6], 0.0).reshape(-1)
    return [out]
