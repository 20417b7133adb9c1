"""GPU: the autotuner keeps what a batch finds.  A wall of many clusters is lit from its own plane;
of the routings, only the built-in and the block path find all of its hits, so a tuned batch has
one of them and the same flags as before, and as the oracle in coherent blocks.
"""
import numpy as np
import pytest

from test_gpu_grazing import W, _coherent, _wall

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 2])
def test_tuned_batch_keeps_grazing_hits(rt, scenes, orc, gpu_ctx, seed):
    v9, u, v = _wall(np.random.default_rng(seed), 40)
    sc = rt.Scene(gpu_ctx, v9, desc="rayhierarchy")
    dev = rt.DeviceRays.from_numpy(scenes.pinhole_rays(W, W, origin=(0, 0, -3.0)))
    hits = sc.trace_closest(dev)
    shadow = rt.make_shadow_rays(dev, hits, tuple(np.float32([0, 0, 2]) + 3 * u + 0.5 * v))
    host = {k: getattr(shadow, k).cpu().numpy()
            for k in ("ox", "oy", "oz", "dx", "dy", "dz", "tmin", "tmax", "valid")}
    host.update(width=W, height=W)
    ref = orc.trace(v9, host, orc.params("rayhierarchy"), orc.OCCLUDED)["occ"]
    b = rt.Batch(gpu_ctx)
    h, occ = b.add_closest(sc, dev), b.add_occluded(sc, shadow)
    check = _coherent(host, 3)
    for tuned in (False, True):
        if tuned:
            b.autotune(reps=2)
            for p in (rt.RT_PARAM_RAY_CLUSTERS_CLOSEST, rt.RT_PARAM_RAY_CLUSTERS_OCCLUDED):
                assert b.get_param(p) in (0, rt.RAY_PATH_OFF)
        occ.fill_(7)
        b.run()
        assert np.array_equal(occ.cpu().numpy()[check], ref[check])
        assert np.array_equal(h.id.cpu().numpy(), hits.id.cpu().numpy())
    assert ref[check].sum() > 0
    b.close()
    sc.close()
