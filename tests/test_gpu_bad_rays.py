"""GPU: rays that are not finite, or start absurdly far away, beside ordinary ones.

Such a ray passes every plane test of the search tree and walks all of it.  The bad rays fill
whole blocks of the image, so that no hierarchy node mixes them with ordinary rays: those have to
come out bit for bit as in an image without any bad ray.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W, H, B = 96, 64, 16  # B: block side of 4x4 leaves and three levels


@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_ordinary_rays_unchanged(rt, scenes, gpu_ctx, accel):
    v9 = scenes.room_scene(seed=3, nclusters=400)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel))
    good = scenes.pinhole_rays(W, H, origin=(0.0, 0.0, -9.0), fov_deg=50.0)
    seg = scenes.random_rays(W * H, seed=4, lo=-4.0, hi=4.0, maxt=6.0, width=W)
    blk = (np.arange(W * H) // W // B + np.arange(W * H) % W // B) % 3 == 1
    at = np.flatnonzero(blk)
    kind = np.arange(len(at)) // 2 % 6  # neighbours of each kind, so lanes of every kind meet
    for mode, src in ((0, good), (1, seg), (2, seg)):
        bad = {k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in src.items()}
        with np.errstate(over="ignore"):
            for a, k in enumerate(("x", "y", "z")):
                o, d = bad["o" + k], bad["d" + k]
                d[at[kind == 0]] = np.nan
                o[at[kind == 1]] = np.nan
                d[at[kind == 2]] = np.inf
                o[at[kind == 3]] = -np.inf
                for q, far in ((4, 1e9), (5, 1e30)):
                    o[at[kind == q]] = far
                    d[at[kind == q]] = -0.57735026
        out = []
        for r in (src, bad):
            print(f"[bad rays] {accel} mode {mode} {'bad' if r is bad else 'plain'}", flush=True)
            dev = rt.DeviceRays.from_numpy(r)
            if mode == 2:
                out.append([sc.trace_occluded(dev).cpu().numpy()])
            else:
                h = sc.trace_closest(dev, mode)
                out.append([x.cpu().numpy() for x in (h.id, h.t, h.u, h.v)])
        for k, (x, y) in enumerate(zip(*out)):
            assert np.array_equal(x[~blk].view(np.uint8), y[~blk].view(np.uint8)), \
                f"mode {mode}: output {k} of ordinary rays differs"
        assert (out[0][0][~blk] > 0).sum() > 100
        if mode < 2:  # the strict test never accepts a ray that is not finite
            assert (out[1][0][at[kind < 4]] == -1).all()
    sc.close()
