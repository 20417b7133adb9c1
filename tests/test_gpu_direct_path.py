"""GPU: the built-in routing, in which the per-ray kernel itself writes misses, records, flags and
the list of rays to repair, over the cases where that can go wrong: chains that fail for no, some
or all strict hits, with a full queue (one wavefront for the whole image) and rays that find no
room in it; trees with absent children, median splits and deep nodes; rays from far outside; and
few rays whose subtrees idle lanes take over.

The default is compared with the block path (every candidate enumerated) bit for bit, and images
of many jobs in one launch with the same jobs alone.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _force(rt, b, threshold, grid=0):
    for p in (rt.RT_PARAM_RAY_CLUSTERS_CLOSEST, rt.RT_PARAM_RAY_CLUSTERS_OCCLUDED):
        b.set_param(p, threshold)
    for p in (rt.RT_PARAM_RAY_GRID_CLOSEST, rt.RT_PARAM_RAY_GRID_OCCLUDED):
        b.set_param(p, grid)


def _run(rt, ctx, sc, dev, mode, threshold, grid=0, copies=1):
    """Outputs of `copies` equal closest and occlusion jobs in one batch."""
    b = rt.Batch(ctx)
    _force(rt, b, threshold, grid)
    jobs = [(b.add_closest(sc, dev, mode), b.add_occluded(sc, dev)) for _ in range(copies)]
    for h, occ in jobs:     # nothing of an earlier run may pass for a result
        for x in (h.id, h.t, h.u, h.v, occ):
            x.fill_(77)
    b.run()
    out = [[x.cpu().numpy() for x in (h.id, h.t, h.u, h.v, occ)] for h, occ in jobs]
    b.close()
    return out


def _same(got, want, what):
    for k, (x, y) in enumerate(zip(got, want)):
        m = int((x.view(np.uint8) != y.view(np.uint8)).sum())
        assert m == 0, f"{what}: {m} bytes of output {k} differ"


def _failing(scenes, share, w, h):
    """Rays going down; `share` of them with directions five times unit length, whose chains fail
    by the raw d.z of node box_uv."""
    v9 = scenes.random_triangles(3000, seed=2, extent=1.0, size=0.15)
    g = np.random.default_rng(4)
    n = w * h
    d = g.normal(size=(n, 3)) * [1.0, 0.2, 1.0] + [0.0, -2.0, 0.0]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d *= np.where(g.random(n) < share, 5.0, 1.0)[:, None]
    o = g.uniform(-0.8, 0.8, size=(n, 3)) + [0.0, 2.0, 0.0]
    rays = {k: np.ascontiguousarray(a, np.float32)
            for k, a in zip(("ox", "oy", "oz", "dx", "dy", "dz"), (*o.T, *d.T))}
    rays.update(tmin=np.zeros(n, np.float32), tmax=np.full(n, 3.0, np.float32), valid=None,
                width=w, height=h)
    return v9, rays


@pytest.mark.parametrize("w,h,copies", [(64, 48, 1), (64, 48, 3), (5, 3, 1), (400, 300, 1)])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0], ids=lambda s: f"failing{s}")
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_failing_chains(rt, scenes, gpu_ctx, accel, share, w, h, copies):
    v9, rays = _failing(scenes, share, w, h)
    dev = rt.DeviceRays.from_numpy(rays)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel, node="box_uv"))
    for mode in (rt.RT_CLOSEST_PRIMARY, rt.RT_CLOSEST_SECONDARY):
        print(f"[direct] {accel} share {share} {w}x{h} x{copies} mode {mode}", flush=True)
        block = _run(rt, gpu_ctx, sc, dev, mode, rt.RAY_PATH_OFF)[0]
        for grid in (0, 1):
            for got in _run(rt, gpu_ctx, sc, dev, mode, 0, grid, copies):
                _same(got, block, f"grid {grid}")
        if share == 0.0:
            assert (block[0] >= 0).sum() > w * h // 4
    sc.close()


def _shape(name, scenes):
    g = np.random.default_rng(5)
    if name[1:].isdigit():
        return scenes.random_triangles(int(name[1:]), seed=3, size=0.6)
    if name == "identical":
        return np.tile(scenes.random_triangles(1, seed=3, extent=0.0, size=0.8), (300, 1))
    if name == "geometric":
        s = (1.02 ** -np.arange(1200))[:, None].astype(np.float32)
        return (scenes.random_triangles(1200, seed=4, extent=0.2, size=0.8) * s).astype(np.float32)
    assert name == "offset"
    return (scenes.random_triangles(500, seed=7, size=0.3)
            + np.tile(np.float32([4096, -2048, 0]), 3)).astype(np.float32)


@pytest.mark.parametrize("name", ["n1", "n2", "n3", "n4", "n5", "n17", "n65", "identical",
                                  "geometric", "offset"])
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_trees(rt, scenes, gpu_ctx, name, accel):
    v9 = _shape(name, scenes)
    c = v9.reshape(-1, 3).mean(0)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel, node="ia"))
    far = scenes.pinhole_rays(48, 32, origin=tuple(c + [0, 0, -900.0]), fov_deg=0.2)
    rnd = scenes.random_rays(48 * 32, seed=10, lo=-1.5, hi=1.5, maxt=np.inf, width=48)
    for k, x in zip(("ox", "oy", "oz"), c):
        rnd[k] = (rnd[k] + np.float32(x)).astype(np.float32)
    hits = 0
    for rays, mode in ((scenes.pinhole_rays(48, 32, origin=tuple(c + [0, 0, -3.0])), 0), (far, 0),
                       (rnd, 1)):
        dev = rt.DeviceRays.from_numpy(rays)
        print(f"[direct] {accel} {name} mode {mode}", flush=True)
        block = _run(rt, gpu_ctx, sc, dev, mode, rt.RAY_PATH_OFF)[0]
        for grid in (0, 1):
            _same(_run(rt, gpu_ctx, sc, dev, mode, 0, grid)[0], block, f"{name} grid {grid}")
        hits += int((block[0] >= 0).sum())
    assert hits > 0
    sc.close()


@pytest.mark.parametrize("array", ["ox", "dz", "tmin", "tmax"])
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_distances_over_the_rays(rt, scenes, gpu_ctx, accel, array):
    """A ray's record is written when nothing of the ray is needed any more, so distances may
    replace one of the rays' own arrays."""
    v9, rays = _failing(scenes, 0.3, 64, 48)
    dev = rt.DeviceRays.from_numpy(rays)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel, node="box_uv"))
    mode = rt.RT_CLOSEST_SECONDARY
    apart = sc.trace_closest(dev, mode)
    over = rt.DeviceHits.empty(dev.count)
    over.t = getattr(dev, array)
    sc.trace_closest(dev, mode, hits=over)
    _same([getattr(over, k).cpu().numpy() for k in ("id", "t", "u", "v")],
          [getattr(apart, k).cpu().numpy() for k in ("id", "t", "u", "v")], array)
    assert (apart.id.cpu().numpy() >= 0).sum() > 100
    sc.close()


@pytest.mark.parametrize("scale", [1e-20, 1e-37, 2e-38])
@pytest.mark.parametrize("node", ["box_dir", "box_uv", "ia"])
def test_infinite_distances(rt, scenes, gpu_ctx, node, scale):
    """Directions so short that the distance of a hit overflows: the leaf test passes, the hit is
    no nearest one, but the repair pass takes it where a primary ray has no other."""
    v9 = (scenes.random_triangles(300, seed=3, size=0.6) * 4).astype(np.float32)
    rays = scenes.pinhole_rays(48, 32, origin=(0, 0, -12.0))
    for k in ("dx", "dy", "dz"):
        rays[k] = (rays[k] * np.float32(scale)).astype(np.float32)
    rays["dz"][::3] *= np.float32(50)       # with scale 2e-38, some whose distances are finite
    dev = rt.DeviceRays.from_numpy(rays)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc("rayhierarchy", node=node))
    for mode in (0, 1):
        print(f"[direct] infinite distances {node} {scale} mode {mode}", flush=True)
        block = _run(rt, gpu_ctx, sc, dev, mode, rt.RAY_PATH_OFF)[0]
        far = int(((block[0] >= 0) & np.isinf(block[1])).sum())
        print(f"[direct] {far} at an infinite distance, {int((block[0] >= 0).sum())} hits", flush=True)
        assert (far > 0) == (mode == 0 and scale == 2e-38)
        _same(_run(rt, gpu_ctx, sc, dev, mode, 0)[0], block, node)
    sc.close()
