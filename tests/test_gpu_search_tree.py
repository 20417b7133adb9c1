"""GPU: the per-ray path's 4-wide search tree at the sizes and shapes where it can go wrong.

The tree only narrows which triangles a ray tests, so a trace that takes it must equal the block
path, which enumerates every candidate, bit for bit: scenes of one to a few triangles (absent
children), coinciding triangles (median splits), sizes shrinking geometrically (deep binary
trees, where nodes keep fewer children so that the walk's stack fits), scenes far from the
origin, rays parallel to the axes and origins far outside.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(name, scenes):
    g = np.random.default_rng(5)
    if name[1:].isdigit():
        return scenes.random_triangles(int(name[1:]), seed=3, size=0.6)
    if name == "identical":
        return np.tile(scenes.random_triangles(1, seed=3, extent=0.0, size=0.8), (300, 1))
    if name == "geometric":
        s = (1.02 ** -np.arange(1200))[:, None].astype(np.float32)
        return (scenes.random_triangles(1200, seed=4, extent=0.2, size=0.8) * s).astype(np.float32)
    if name == "offset":
        return (scenes.random_triangles(500, seed=7, size=0.3)
                + np.tile(np.float32([4096, -2048, 0]), 3)).astype(np.float32)
    assert name == "flat"
    v = scenes.random_triangles(500, seed=8, size=0.3)
    v[:, 2::3] = g.choice([0.0, 0.5], size=(500, 1)).astype(np.float32)
    return v


def _rays(name, v9, kind, scenes):
    c = v9.reshape(-1, 3).mean(0)
    if kind == "camera":
        return scenes.pinhole_rays(48, 32, origin=tuple(c + [0, 0, -3.0]))
    if kind == "far":
        return scenes.pinhole_rays(48, 32, origin=tuple(c + [0, 0, -900.0]), fov_deg=0.2)
    g = np.random.default_rng(9)
    r = scenes.random_rays(48 * 32, seed=10, lo=-1.5, hi=1.5, maxt=np.inf, width=48)
    for k, x in zip(("ox", "oy", "oz"), c):
        r[k] = (r[k] + np.float32(x)).astype(np.float32)
    # a third of the directions along an axis, with zeros of either sign
    ax = g.integers(0, 9, size=48 * 32)
    for k, a in zip(("dx", "dy", "dz"), range(3)):
        r[k] = np.where(ax == a, np.float32(1), np.where(ax < 3, g.choice(np.float32([0.0, -0.0]), 48 * 32),
                                                        r[k])).astype(np.float32)
    return r


SHAPES = ["n1", "n2", "n3", "n4", "n5", "n6", "n17", "n65", "identical", "geometric", "offset",
          "flat"]


def _traced(sc, d, mode):
    import torch
    h = sc.trace_closest(d, mode)
    return [x.cpu().numpy() for x in (h.id, h.t.view(torch.int32), h.u.view(torch.int32),
                                      h.v.view(torch.int32), sc.trace_occluded(d))]


def _force(rt, sc, threshold):
    sc.set_param(rt.RT_PARAM_RAY_CLUSTERS_CLOSEST, threshold)
    sc.set_param(rt.RT_PARAM_RAY_CLUSTERS_OCCLUDED, threshold)


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_wide_tree_equals_enumeration(rt, scenes, gpu_ctx, name, accel):
    v9 = _scene(name, scenes)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel, node="ia"))
    hits = 0
    for kind, mode in (("camera", 0), ("far", 0), ("random", 1)):
        print(f"[search tree] {accel} {name} {kind}", flush=True)
        d = rt.DeviceRays.from_numpy(_rays(name, v9, kind, scenes))
        _force(rt, sc, 1)
        ray = _traced(sc, d, mode)
        _force(rt, sc, rt.RAY_PATH_OFF)
        for k, (a, b) in enumerate(zip(ray, _traced(sc, d, mode))):
            n = int((a != b).sum())
            assert n == 0, f"{accel} {name} {kind}: {n} mismatches in output {k}"
        hits += int((ray[0] >= 0).sum())
    assert hits > 0
    sc.close()
