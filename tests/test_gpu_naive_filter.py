"""GPU: the naive accelerator over the ways its work-groups split rays and triangles (one ray, odd
counts, triangles that do not fill or just overfill a staged group) and over the geometry its
filter has to let through: edges and corners hit exactly, rays in a triangle's plane, zero
determinants, magnitudes from 1e-18 to 1e18, infinities and NaN.  Ids, t and flags are the
oracle's, bit for bit up to the sign of a zero t.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(rng, ntri, scale):
    v9 = rng.uniform(-1, 1, (ntri, 3, 3))
    v9[1::7, 2] = v9[1::7, 1]                       # no area
    v9[2::7, :, 2] = 0.25                           # in a plane of constant z
    v9[3::7] = np.round(v9[3::7] * 4) / 4           # on a grid
    return (v9 * scale).astype(np.float32)


def _rays(rng, v9, w, h, scale):
    n = w * h
    tri = v9[rng.integers(0, len(v9), n)].astype(np.float64)
    b = rng.uniform(-0.2, 1.2, (n, 2))
    b[::3, 0] = rng.choice([0.0, 1.0, -1e-3, 1.001, -0.003, 1.003], len(b[::3]))
    b[1::5, 1] = 1.001 - b[1::5, 0]
    p = tri[:, 0] + b[:, :1] * (tri[:, 1] - tri[:, 0]) + b[:, 1:] * (tri[:, 2] - tri[:, 0])
    o = rng.uniform(-2, 2, (n, 3)) * scale
    o[::4, 2] = 0.25 * scale
    d = p - o
    d[2::9] = tri[2::9, 1] - tri[2::9, 0]           # along an edge
    d[::4, 2] = np.where(np.arange(len(d[::4])) % 2, 0.0, d[::4, 2])
    f = lambda a: np.ascontiguousarray(a, np.float32)
    return dict(ox=f(o[:, 0]), oy=f(o[:, 1]), oz=f(o[:, 2]), dx=f(d[:, 0]), dy=f(d[:, 1]),
                dz=f(d[:, 2]), tmin=np.zeros(n, np.float32), tmax=np.full(n, 1.5, np.float32),
                valid=(rng.random(n) < 0.9).astype(np.uint8), width=w, height=h)


@pytest.mark.parametrize("ntri,w,h,scale", [(1, 1, 1, 1.0), (5, 31, 7, 1.0), (511, 64, 33, 1.0),
                                            (513, 40, 9, 1e4), (1025, 129, 65, 1.0),
                                            (70, 300, 220, 0.01), (9, 400, 330, 1.0), (300, 50, 20, 1e18),
                                            (300, 50, 20, 1e-18), (200, 37, 11, 1e12)])
def test_naive_equals_oracle(rt, orc, gpu_ctx, ntri, w, h, scale):
    rng = np.random.default_rng(ntri * 1000 + w)
    v9 = _scene(rng, ntri, scale)
    rays = _rays(rng, v9, w, h, scale)
    p = orc.params("naive")
    for bad in (False, True):
        if bad:  # occlusion only: the key of a NaN distance is the reduction's own order
            rays["ox"][::17], rays["dy"][1::19], rays["dz"][2::23] = np.inf, np.nan, -np.inf
            if ntri > 20:
                v9[5, 1, 0], v9[11, 2, 1], v9[17, 0, 2] = np.inf, np.nan, -np.inf
        sc = rt.Scene(gpu_ctx, v9, desc="naive")
        d = rt.DeviceRays.from_numpy(rays)
        for mode in ((2,) if bad else (0, 1, 2)):
            print(f"[naive] {ntri} triangles {w}x{h} scale {scale} mode {mode} {bad}", flush=True)
            ref = orc.trace(v9, rays, p, mode if mode < 2 else orc.OCCLUDED)
            if mode == 2:
                assert np.array_equal(sc.trace_occluded(d).cpu().numpy(), ref["occ"])
            else:
                hit = sc.trace_closest(d, mode)
                assert np.array_equal(hit.id.cpu().numpy(), ref["id"])
                k = ref["id"] >= 0
                zero = np.float32(0)  # the reduction key makes a hit at -0 one at +0
                assert np.array_equal((hit.t.cpu().numpy()[k] + zero).view(np.uint32),
                                      (ref["t"][k] + zero).view(np.uint32))
        sc.close()
