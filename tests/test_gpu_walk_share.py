"""GPU: RT_PARAM_WALK_* v stands for 1/2^v of the lanes whatever the built-in share is.  Results
are the same for every value; the share itself is seen in the library's source, whose table the
kernel launch reads.
"""
import re
from pathlib import Path

import numpy as np
import pytest

SRC = Path(__file__).resolve().parent.parent / "pbrt-v2_amd" / "csrc" / "rt_kernels.hip"


def test_shares():
    m = re.search(r"kWalk64\[8\] = \{([^}]*)\}", SRC.read_text())
    share = [int(x) / 64 for x in m.group(1).split(",")]
    assert share[0] == 3 / 8
    assert share[1:7] == [0.5 ** v for v in range(1, 7)] and share[7] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_results_for_every_share(rt, scenes, gpu_ctx, accel):
    v9 = scenes.random_triangles(2000, seed=3, size=0.2)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(accel))
    dev = rt.DeviceRays.from_numpy(scenes.pinhole_rays(64, 48, origin=(0, 0, -3.0)))
    want = None
    for v in range(8):
        for p in (rt.RT_PARAM_WALK_CLOSEST, rt.RT_PARAM_WALK_OCCLUDED):
            sc.set_param(p, v)
        h, occ = sc.trace_closest(dev), sc.trace_occluded(dev)
        got = [x.cpu().numpy() for x in (h.id, h.t, h.u, h.v, occ)]
        want = want or got
        assert all(np.array_equal(a.view(np.uint8), b.view(np.uint8)) for a, b in zip(got, want)), v
    assert (want[0] >= 0).any()
    sc.close()
