"""CPU: the per-ray path's search tree as the product builds it, walked on the host with the
kernel's node test (tests/cpp/search_walk.cpp).

The walk's stack in LDS has a fixed number of entries and no check: the tree has to fit it for
every ray there can be, also for directions or origins that are not finite and origins so far out
that every plane test passes.
"""
import ctypes
from pathlib import Path

import numpy as np
import pytest

LIB = Path(__file__).resolve().parent / "cpp" / "libsearch_walk.so"


class Walk:
    def __init__(self, v9):
        if not LIB.exists():
            pytest.fail(f"{LIB} is not built (run __graft_entry__.build())")
        self.lib = ctypes.CDLL(str(LIB))
        self.lib.sw_build.restype = ctypes.c_void_p
        v9 = np.ascontiguousarray(v9, np.float32).reshape(-1, 9)
        self.ntri = len(v9)
        self.h = ctypes.c_void_p(self.lib.sw_build(ctypes.c_void_p(v9.ctypes.data),
                                                   ctypes.c_uint32(self.ntri)))
        self.stack = self.lib.sw_stack()

    def walk(self, rays, every=False):
        """rays: (n, 8) origin, direction, interval -> stack entries, nodes, triangles per ray."""
        with np.errstate(over="ignore"):
            r = np.ascontiguousarray(rays, np.float32).reshape(-1, 8)
        out = [np.zeros(len(r), np.int32), np.zeros(len(r), np.uint32), np.zeros(len(r), np.uint32)]
        self.lib.sw_walk(self.h, ctypes.c_void_p(r.ctypes.data), ctypes.c_uint32(len(r)),
                         ctypes.c_int(int(every)),
                         *(ctypes.c_void_p(a.ctypes.data) for a in out), None)
        return out

    def close(self):
        self.lib.sw_free(self.h)


def _bad_rays(scale):
    nan, inf = np.nan, np.inf
    o, d = [0.1, 0.2, -0.3], [0.3, -0.5, 0.8]
    rays = [[nan] * 3 + d, [inf] * 3 + d, [-inf, inf, -inf] + d, o + [nan] * 3, o + [inf] * 3,
            o + [-inf, inf, inf], [nan] * 3 + [inf] * 3, o + [0.0] * 3, [nan, 0, 0] + d,
            o + [inf, 0.0, -0.0]]
    for far in (1e9, 1e10, 1e20, 3e38):
        p = np.array([far, far, far]) * scale
        with np.errstate(over="ignore"):
            rays.append([*p, *(-p / np.linalg.norm(p))])
            rays.append([*p, -1.0, -1.0, -1.0])
    return np.array([r + t for r in rays for t in ([0.0, inf], [nan, nan], [-inf, inf], [inf, 1.0])])


@pytest.mark.parametrize("name", ["clusters200k", "clusters100k", "room80k", "geometric", "same"])
def test_walk_fits_its_stack(scenes, name):
    if name.startswith("clusters"):
        v9 = scenes.cluster_scene(200000 if "200" in name else 100000, seed=1)
    elif name == "room80k":
        v9 = scenes.room_scene(seed=3, nclusters=400)
    elif name == "geometric":
        s = (1.02 ** -np.arange(4000))[:, None].astype(np.float32)
        v9 = (scenes.random_triangles(4000, seed=4, extent=0.2, size=0.8) * s).astype(np.float32)
    else:
        v9 = np.tile(scenes.random_triangles(1, seed=3, extent=0.0, size=0.8), (5000, 1))
    w = Walk(v9)
    one = [[0.0] * 3 + [0.0, 0.0, 1.0] + [0.0, np.inf]]
    depth, _, leaves = w.walk(one, every=True)
    assert leaves[0] == w.ntri  # the tree holds every triangle once
    assert depth[0] <= w.stack
    depth, visits, _ = w.walk(_bad_rays(float(np.abs(v9).max())))
    assert depth.max() <= w.stack
    g = np.random.default_rng(0)
    rnd = np.concatenate([g.uniform(-5, 5, (2000, 3)), g.normal(size=(2000, 3)),
                          np.tile([0.0, np.inf], (2000, 1))], axis=1)
    assert w.walk(rnd)[0].max() <= w.stack
    w.close()
