"""GPU: hierarchy builds over leaf sizes around the lanes a leaf is shared by (one ray, powers of
two, one off them, more than 64 rays, more than 64 * 4), images that the leaves do not divide, and
rays that are not valid.  The nodes show in the cull chains, so hits and occlusion are compared
with the oracle's; box_dir's culls depend on every bound of a node.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cx,cy,height", [(1, 1, 3), (2, 1, 3), (3, 1, 2), (3, 5, 2), (4, 4, 3),
                                          (17, 1, 2), (9, 7, 2), (8, 8, 2), (13, 5, 1), (16, 8, 2),
                                          (100, 4, 2), (7, 41, 1), (4, 2, 6)])
def test_leaf_sizes(rt, scenes, orc, gpu_ctx, cx, cy, height):
    v9 = scenes.random_triangles(300, seed=5, size=0.35)
    g = np.random.default_rng(cx * 100 + cy)
    for node in ("box_dir", "box_uv"):
        sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc("rayhierarchy", node=node, chunk_x=cx,
                                                        chunk_y=cy, height=height))
        p = orc.params("rayhierarchy", node=node, cx=cx, cy=cy, height=height)
        cam = scenes.pinhole_rays(75, 43)
        rnd = scenes.random_rays(75 * 43, seed=cy, lo=-1.0, hi=1.0, maxt=2.0, width=75)
        rnd["valid"] = (g.random(75 * 43) < 0.7).astype(np.uint8)
        rnd["dx"][::9] = 0.0  # the validity-aware 5DB build restarts a slope there
        for mode, rays in ((0, cam), (1, rnd), (2, rnd)):
            print(f"[leaf build] {cx}x{cy} height {height} {node} mode {mode}", flush=True)
            d = rt.DeviceRays.from_numpy(rays)
            ref = orc.trace(v9, rays, p, mode if mode < 2 else orc.OCCLUDED)
            if mode == 2:
                assert np.array_equal(sc.trace_occluded(d).cpu().numpy(), ref["occ"])
            else:
                h = sc.trace_closest(d, mode)
                assert np.array_equal(h.id.cpu().numpy(), ref["id"])
                hit = ref["id"] >= 0
                assert np.array_equal(h.t.cpu().numpy()[hit].view(np.uint32),
                                      ref["t"][hit].view(np.uint32))
        sc.close()
