"""CPU: which strict hits the search tree may miss, with the product's builder and bounds
(tests/cpp/search_walk.cpp).

The strict leaf test accepts a ray close to a triangle's plane by its roundings, where no padded
box is.  Every strict hit has to be reached by the walk or be one that the grazing pass's bounds
let through, for the ray alone and for the boxes of a group of rays.
"""
import ctypes

import numpy as np
import pytest

from test_search_tree import Walk


def _check(w, rays, group=16):
    r = np.ascontiguousarray(rays, np.float32)
    out = np.zeros(6, np.uint64)
    w.lib.sw_grazing(w.h, ctypes.c_void_p(r.ctypes.data), ctypes.c_uint32(len(r)),
                     ctypes.c_uint32(group), ctypes.c_void_p(out.ctypes.data))
    hits, missed, lost, lost_group, pairs, _ = (int(x) for x in out)
    assert lost == 0, f"{lost} of {hits} strict hits neither reached nor taken for grazing"
    assert lost_group == 0, f"{lost_group} of {hits} by the boxes of {group} rays"
    return hits, missed, pairs


def _grazing_rays(g, v9, n, spread):
    """Rays toward points in and around the planes of the triangles, at angles down to zero."""
    t = v9.reshape(-1, 3, 3).astype(np.float64)[g.integers(0, len(v9), n)]
    e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    nn = np.cross(e1, e2)
    nn = nn / np.maximum(np.linalg.norm(nn, axis=1, keepdims=True), 1e-300)
    a = e1 / np.maximum(np.linalg.norm(e1, axis=1, keepdims=True), 1e-30)
    b = np.cross(nn, a)
    th = g.uniform(0, 2 * np.pi, (n, 1))
    al = 10.0 ** g.uniform(-9, -1, (n, 1)) * g.choice([-1, 1], (n, 1))
    al[::3] = 0
    d = np.cos(th) * a + np.sin(th) * b + al * nn
    bb = g.uniform(-0.3, 1.3, (n, 2))
    p = t[:, 0] + bb[:, :1] * e1 + bb[:, 1:] * e2
    p = p + g.normal(size=(n, 3)) * 10.0 ** g.uniform(-9, 0, (n, 1)) * (g.random((n, 1)) < 0.5)
    s = g.uniform(0, spread, (n, 1))
    o = p - s * d
    d = d * np.where(g.random((n, 1)) < 0.3, 10.0 ** g.uniform(-3, 3, (n, 1)), 1.0)
    tmax = np.where(g.random(n) < 0.5, np.inf, g.uniform(0, 2, n) * s[:, 0])
    return np.concatenate([o, d, np.zeros((n, 1)), tmax[:, None]], 1)


def _scene(name, scenes, g):
    soup = scenes.random_triangles(300, seed=1, size=0.3)
    if name == "soup":
        return soup
    if name == "small":
        return scenes.random_triangles(300, seed=1, size=0.02)
    if name == "offset":
        return soup + np.tile(np.float32([4096, -2048, 100]), 3)
    if name == "big":
        return soup * np.float32(1e6)
    if name == "tiny":
        return soup * np.float32(1e-4)
    if name == "flat":
        v = soup.copy()
        v[:, 2::3] = g.choice([0, 0.5], (300, 1)).astype(np.float32)
        return v
    if name == "room":
        return scenes.room_scene(seed=3, nclusters=2)
    if name == "clusters":
        return scenes.cluster_scene(400, seed=2)
    t = soup.reshape(-1, 3, 3).copy()
    t[:, 2] = t[:, 1] + (t[:, 2] - t[:, 1]) * (10.0 ** g.uniform(-8, 0, (300, 1))).astype(np.float32)
    if name == "degenerate":
        t[::2, 2] = t[::2, 1]
        t[1::8, 1] = t[1::8, 0]
    else:
        assert name == "thin"
    return t.reshape(-1, 9)


@pytest.mark.parametrize("name", ["soup", "small", "offset", "big", "tiny", "flat", "room",
                                  "clusters", "thin", "degenerate"])
def test_every_strict_hit_is_accounted_for(scenes, name):
    g = np.random.default_rng(7)
    v9 = np.ascontiguousarray(_scene(name, scenes, g), np.float32)
    w = Walk(v9)
    ext = float(np.ptp(v9.reshape(-1, 3), axis=0).max())
    hits = 0
    for spread in (2, 30, 1000):
        hits += _check(w, _grazing_rays(g, v9, 2000, spread * ext / 2))[0]
    c = v9.reshape(-1, 3).mean(0)
    o = c + g.normal(size=(2000, 3)) * ext
    rnd = np.concatenate([o, g.normal(size=(2000, 3)), np.zeros((2000, 1)),
                          np.full((2000, 1), np.inf)], 1)
    hits += _check(w, rnd)[0]
    assert hits > 100
    w.close()


@pytest.mark.parametrize("k", [2, 20])
def test_light_in_the_plane_of_a_wall(scenes, k):
    # shadow rays of a rotated wall toward lights in its own plane: the tree alone misses some
    missed = hits = 0
    for seed in range(6):
        g = np.random.default_rng(seed)
        u, v, n = np.linalg.qr(g.normal(size=(3, 3)))[0]
        a = (2.0 * np.arange(k + 1) / k - 1.0) * 2.0
        p = np.array([0, 0, 2.0]) + a[:, None, None] * u + a[None, :, None] * v
        q = [p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]]
        v9 = np.stack([np.stack([q[0], q[1], q[2]], 2), np.stack([q[0], q[2], q[3]], 2)],
                      2).reshape(-1, 9).astype(np.float32)
        ab = g.uniform(-2, 2, (1500, 2))
        o = (np.array([0, 0, 2.0]) + ab[:, :1] * u + ab[:, 1:] * v).astype(np.float32)
        light = np.array([0, 0, 2.0]) + u * 3.0 + v * g.uniform(-3, 3)
        d = light - o
        dist = np.linalg.norm(d, axis=1, keepdims=True)
        w = Walk(v9)
        h, m, _ = _check(w, np.concatenate([o, d / dist, np.full((1500, 1), 1e-3),
                                            dist * 0.999], 1))
        hits += h
        missed += m
        w.close()
    assert hits > 100 and missed > 0  # what the pass is for
