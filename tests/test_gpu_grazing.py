"""GPU: rays that run in the plane of a surface, default routing, against the oracle.

The strict leaf test accepts some of them by its roundings alone, anywhere along the plane, where
no padded box is.  A rotated wall lit by a point light in its own plane, or seen edge on by the
camera, has many; thin and degenerate triangles have them at larger angles.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = 96


def _axes(g):
    q, _ = np.linalg.qr(g.normal(size=(3, 3)))
    return q


def _wall(g, k, half=2.0, center=(0.0, 0.0, 2.0)):
    """k x k quads in a random plane through `center`; its triangles and two axes in the plane."""
    u, v, _ = _axes(g)
    a = (2.0 * np.arange(k + 1) / k - 1.0) * half
    p = np.array(center) + a[:, None, None] * u + a[None, :, None] * v
    q = [p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]]
    t = np.stack([np.stack([q[0], q[1], q[2]], 2), np.stack([q[0], q[2], q[3]], 2)], 2)
    return np.ascontiguousarray(t.reshape(-1, 9), np.float32), u, v


def _thin(g, n, dead):
    """Needles of every width, some without any area, around a wall."""
    t = g.uniform(-1.5, 1.5, (n, 1, 3)) + g.normal(size=(n, 3, 3)) * 0.5 + [0, 0, 2.0]
    t[:, 2] = t[:, 1] + (t[:, 2] - t[:, 1]) * 10.0 ** g.uniform(-7, 0, (n, 1))
    if dead:
        t[::3, 2] = t[::3, 1]
    return t.reshape(-1, 9).astype(np.float32)


def _coherent(rays, height):
    """Rays of the blocks whose leaves spread their directions by 0.25 on average at most; the
    others, and the rays that are not traced, are left to the tree alone."""
    b = 4 << (height - 1)
    valid = np.ones(W * W, bool) if rays["valid"] is None else rays["valid"] > 0
    d = np.stack([rays[k] for k in ("dx", "dy", "dz")], 1).reshape(W, W, 3)
    v = valid.reshape(W, W)
    out = np.zeros((W, W), bool)
    for y in range(0, W, b):
        for x in range(0, W, b):
            s = [np.ptp(d[j:j + 4, i:i + 4][v[j:j + 4, i:i + 4]], axis=0).max()
                 for j in range(y, min(y + b, W), 4) for i in range(x, min(x + b, W), 4)
                 if v[j:j + 4, i:i + 4].any()]
            out[y:y + b, x:x + b] = len(s) > 0 and np.mean(s) <= 0.249
    return (out & v).reshape(-1)


def _noalloc(rt, sc, rays):
    h = rt.DeviceHits.empty(rays.count)
    rs, hs = rays.c_struct(), h.c_struct()
    assert rt.lib().rt_trace_closest_noalloc(sc.handle, ctypes.byref(rs), rt.RT_CLOSEST_PRIMARY,
                                             ctypes.byref(hs), None) == 0
    return h


def _check(rt, scenes, orc, ctx, accel, node, v9, origin, light, height=3, least=0):
    sc = rt.Scene(ctx, v9, desc=rt.default_desc(accel, node=node, height=height))
    p = orc.params(accel, node=node, height=height)

    def oracle(rays, mode):
        if accel == "ray-bvh":
            return orc.trace_raybvh(v9, *sc.handoff, rays, p, mode)
        return orc.trace(v9, rays, p, mode)

    cam = scenes.pinhole_rays(W, W, origin=tuple(origin))
    ref = oracle(cam, orc.CLOSEST_PRIMARY)
    dev = rt.DeviceRays.from_numpy(cam)
    hit = ref["id"] >= 0
    for got in (sc.trace_closest(dev), _noalloc(rt, sc, dev)):
        assert np.array_equal(got.id.cpu().numpy(), ref["id"])
        assert np.array_equal(got.t.cpu().numpy()[hit].view(np.uint32), ref["t"][hit].view(np.uint32))
    total = 0
    for lp in light:
        sh = scenes.shadow_rays_np(cam, ref["id"], ref["t"], tuple(lp))
        use = _coherent(sh, height)
        if node == "box_uv":  # its rays count by the range of d.z alone
            use &= _coherent(dict(sh, dx=sh["dz"], dy=sh["dz"]), height)
        d = rt.DeviceRays.from_numpy(sh)
        want = oracle(sh, orc.OCCLUDED)["occ"]
        assert np.array_equal(sc.trace_occluded(d).cpu().numpy()[use], want[use])
        total += int(want[use].sum())
        near = oracle(sh, orc.CLOSEST_SECONDARY)["id"]
        got = sc.trace_closest(d, rt.RT_CLOSEST_SECONDARY)
        assert np.array_equal(got.id.cpu().numpy()[use], near[use])
        b = rt.Batch(ctx)
        out, occ = b.add_closest(sc, dev), b.add_occluded(sc, d)
        b.run()
        assert np.array_equal(out.id.cpu().numpy(), ref["id"])
        assert np.array_equal(occ.cpu().numpy()[use], want[use])
        b.close()
    assert total >= least
    sc.close()


@pytest.mark.parametrize("k", [2, 30])
@pytest.mark.parametrize("node", ["box_dir", "ia", "box_uv"])
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_light_in_the_plane_of_a_wall(rt, scenes, orc, gpu_ctx, accel, node, k):
    for seed in range(3):
        print(f"[grazing] {accel} {node} {k}x{k} wall {seed}", flush=True)
        g = np.random.default_rng(seed)
        v9, u, v = _wall(g, k)
        lights = [np.array([0, 0, 2.0]) + u * a + v * b for a, b in g.uniform(-4, 4, (3, 2))]
        _check(rt, scenes, orc, gpu_ctx, accel, node, v9, (0.0, 0.0, -3.0), lights)


@pytest.mark.parametrize("height", [1, 3, 4])
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_camera_in_the_plane_of_a_wall(rt, scenes, orc, gpu_ctx, accel, height):
    g = np.random.default_rng(11)
    for k in (1, 9):
        print(f"[grazing] {accel} height {height} edge on {k}", flush=True)
        # a vertical and a horizontal wall through the camera, and something behind them
        v9, u, v = _wall(g, k)
        for a in (u, v):
            o = np.array([0, 0, 2.0]) + a * 4.0
            o[2] = min(o[2], -1.0)
            w, wu, wv = _wall(g, k, center=tuple(o))
            both = np.concatenate([w, v9, scenes.random_triangles(200, seed=k, extent=1.5, size=0.5)])
            _check(rt, scenes, orc, gpu_ctx, accel, "box_dir", both, o, [o + wu, o + wv],
                   height=height, least=1)


@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
@pytest.mark.parametrize("dead", [False, True], ids=["thin", "degenerate"])
def test_thin_triangles(rt, scenes, orc, gpu_ctx, accel, dead):
    g = np.random.default_rng(5)
    w, u, v = _wall(g, 8)
    v9 = np.concatenate([w, _thin(g, 600, dead)])
    print(f"[grazing] {accel} thin triangles, degenerate {dead}", flush=True)
    _check(rt, scenes, orc, gpu_ctx, accel, "box_dir", v9, (0.0, 0.0, -3.0),
           [(2.0, 2.0, -2.0), np.array([0, 0, 2.0]) + u * 3 + v], least=100)
    _check(rt, scenes, orc, gpu_ctx, accel, "ia", v9, (0.0, 0.0, -300.0), [(0.0, 2.0, -200.0)])
