"""GPU: the per-ray kernel's queue of candidates whose cull chains are evaluated together.

Node "box_uv" keeps the rays' raw d.z but compares it with normalised directions, so rays going
down with directions five times unit length fail the chain of nearly every strict hit: their
rays go to the stack of rays traced again, and with one wavefront for the whole image (grid 1)
queue and stack fill up and rays that find no room trace again at once.  Every mix must equal
the block path bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("share", [0.0, 0.3, 1.0], ids=lambda s: f"failing{s}")
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_failing_chains(rt, scenes, gpu_ctx, accel, share):
    v9 = scenes.random_triangles(3000, seed=2, extent=1.0, size=0.15)
    g = np.random.default_rng(4)
    n = 64 * 48
    d = g.normal(size=(n, 3)) * [1.0, 0.2, 1.0] + [0.0, -2.0, 0.0]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d *= np.where(g.random(n) < share, 5.0, 1.0)[:, None]
    o = g.uniform(-0.8, 0.8, size=(n, 3)) + [0.0, 2.0, 0.0]
    rays = {k: np.ascontiguousarray(a, np.float32)
            for k, a in zip(("ox", "oy", "oz", "dx", "dy", "dz"), (*o.T, *d.T))}
    rays.update(tmin=np.zeros(n, np.float32), tmax=np.full(n, 3.0, np.float32), valid=None,
                width=64, height=48)
    dev = rt.DeviceRays.from_numpy(rays)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel, node="box_uv"))
    for mode in (rt.RT_CLOSEST_PRIMARY, rt.RT_CLOSEST_SECONDARY):
        print(f"[chain queue] {accel} share {share} mode {mode}", flush=True)
        got = {}
        for path, thr, grid in (("block", rt.RAY_PATH_OFF, 0), ("ray", 1, 0), ("one wave", 1, 1)):
            b = rt.Batch(gpu_ctx)
            for p in (rt.RT_PARAM_RAY_CLUSTERS_CLOSEST, rt.RT_PARAM_RAY_CLUSTERS_OCCLUDED):
                b.set_param(p, thr)
            for p in (rt.RT_PARAM_RAY_GRID_CLOSEST, rt.RT_PARAM_RAY_GRID_OCCLUDED):
                b.set_param(p, grid)
            h, occ = b.add_closest(sc, dev, mode), b.add_occluded(sc, dev)
            b.run()
            got[path] = [x.cpu().numpy() for x in (h.id, h.t, h.u, h.v, occ)]
            b.close()
        for path in ("ray", "one wave"):
            for k, (x, y) in enumerate(zip(got[path], got["block"])):
                m = int((x.view(np.uint8) != y.view(np.uint8)).sum())
                assert m == 0, f"{path}: {m} bytes of output {k} differ"
        if share == 0.0:
            assert (got["block"][0] >= 0).sum() > n // 4
    sc.close()
