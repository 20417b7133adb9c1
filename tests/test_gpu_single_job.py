"""GPU: one job's table entry passed with the build launch against the table uploaded for a batch,
with ray buffers and image sizes that change from call to call and blocks deeper than the LDS
build takes.  Results are whole numbers and bit patterns: they have to be equal.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,node,height", [("rayhierarchy", "box_dir", 1),
                                              ("rayhierarchy", "box_uv", 3),
                                              ("rayhierarchy", "ia", 6),
                                              ("ray-bvh", "box_dir", 3), ("ray-bvh", "ia", 2)])
def test_single_job_equals_batch(rt, scenes, gpu_ctx, kind, node, height):
    v9 = scenes.random_triangles(400, seed=11, size=0.3)
    sc = rt.Scene(gpu_ctx, v9, desc=rt.default_desc(kind, node=node, height=height))
    for turn, (w, h) in enumerate([(64, 48), (33, 17), (64, 48), (1, 1), (150, 9)]):
        rnd = scenes.random_rays(w * h, seed=turn, lo=-1.0, hi=1.0, maxt=2.0, width=w)
        rnd["valid"] = (np.arange(w * h) % 3 != 0).astype(np.uint8)
        for mode in (0, 1, 2):
            print(f"[single job] {kind} {node} {w}x{h} mode {mode}", flush=True)
            d = rt.DeviceRays.from_numpy(rnd)
            b = rt.Batch(gpu_ctx)
            if mode == 2:
                want = b.add_occluded(sc, d)
                b.run()
                assert torch.equal(sc.trace_occluded(d), want)
            else:
                want = b.add_closest(sc, d, mode)
                b.run()
                got = sc.trace_closest(d, mode)
                assert torch.equal(got.id, want.id)
                hit = want.id >= 0
                assert torch.equal(got.t[hit].view(torch.int32), want.t[hit].view(torch.int32))
            torch.cuda.synchronize()
            b.close()
    sc.close()
