"""GPU: naive calls of few rays against many triangles, whose triangles several work-groups share
out: counts around the sizes where the rule begins and ends (1, 2, 9 rays, 1,023 and 1,024 groups
of eight, the least triangles that are shared out and one fewer), nearest hits in any share, rays
that miss, invalid rays, ties between shares, flags written over the rays' own.  Ids, t and flags are the oracle's, bit for bit up to the sign of a zero t.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(ntri, w, h):
    rng = np.random.default_rng(ntri + 7 * w)
    n = w * h
    c = rng.uniform(-1, 1, (ntri, 1, 3))
    v9 = (c + rng.normal(size=(ntri, 3, 3)) * 0.15).astype(np.float32)
    v9[-1] = v9[0]                                   # a tie between the first and the last share
    aim = v9[rng.integers(0, ntri, n)].mean(1)
    aim[::4] = v9[0].mean(0)
    o = rng.uniform(-3, 3, (n, 3))
    d = aim - o
    d[1::5] = -d[1::5]                               # most of these miss
    f = lambda a: np.ascontiguousarray(a, np.float32)
    return v9, dict(ox=f(o[:, 0]), oy=f(o[:, 1]), oz=f(o[:, 2]), dx=f(d[:, 0]), dy=f(d[:, 1]),
                    dz=f(d[:, 2]), tmin=np.zeros(n, np.float32),
                    tmax=np.full(n, 0.7, np.float32),
                    valid=(np.arange(n) % 7 != 3).astype(np.uint8), width=w, height=h)


@pytest.mark.parametrize("ntri,w,h", [(6143, 1, 1), (6144, 1, 1), (6145, 2, 1), (40000, 1, 1),
                                      (40000, 3, 3), (7000, 33, 31), (6145, 88, 93),
                                      (6145, 128, 64), (20001, 11, 13)])
def test_split_equals_oracle(rt, orc, gpu_ctx, ntri, w, h):
    v9, rays = _case(ntri, w, h)
    sc = rt.Scene(gpu_ctx, v9, desc="naive")
    p = orc.params("naive")
    zero = np.float32(0)
    for mode in (0, 1, 2, 0, 2):                     # calls again on the scene's scratch
        print(f"[naive split] {ntri} triangles {w}x{h} mode {mode}", flush=True)
        d = rt.DeviceRays.from_numpy(rays)
        ref = orc.trace(v9, rays, p, mode if mode < 2 else orc.OCCLUDED)
        if mode == 2:
            assert np.array_equal(sc.trace_occluded(d).cpu().numpy(), ref["occ"])
            assert np.array_equal(sc.trace_occluded(d, out=d.valid).cpu().numpy(), ref["occ"])
            continue
        hit = sc.trace_closest(d, mode)
        k = ref["id"] >= 0
        assert np.array_equal(hit.id.cpu().numpy(), ref["id"])
        assert np.array_equal((hit.t.cpu().numpy()[k] + zero).view(np.uint32),
                              (ref["t"][k] + zero).view(np.uint32))
    sc.close()
