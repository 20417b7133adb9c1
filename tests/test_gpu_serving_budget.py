"""GPU: the server charges a request for the scratch that the built-in routing takes: rays, blocks
and hierarchy, not the cluster lists and units of the block path, which grow with the scene.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_requests_share_a_budget(rt, scenes, gpu_ctx, accel):
    """Requests of 128 x 128 rays take 1.34 MB of buffers and at most 0.5 MB of scratch whatever
    the scene, so four of them fit 7.5 MB; with lists and units of 100,000 triangles two did."""
    v9 = scenes.random_triangles(100000, seed=5, size=0.02)
    sc = rt.Scene(gpu_ctx, v9, desc=accel)
    srv = rt.Server(gpu_ctx, [sc], mem_budget=7_500_000, max_active=16)
    try:
        tickets = [srv.submit(0, 128, 128, 1, outputs=False) for _ in range(24)]
        for t in tickets:
            srv.wait(t, timeout_s=60.0)
        ticks, most = srv.counters()
    finally:
        srv.close()
        sc.close()
    print(f"[serve] {accel}: {ticks} ticks, at most {most} requests in one", flush=True)
    assert 3 <= most <= 4
