"""GPU: event times name the kernels that ran: the built-in routing launches no unit kernel and
reports none, the block path does, and the whole covers its parts.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accel", ["rayhierarchy", "ray-bvh"])
def test_unit_kernel_only_where_launched(rt, scenes, gpu_ctx, accel):
    sc = rt.Scene(gpu_ctx, scenes.random_triangles(500, seed=3, size=0.3),
                  desc=rt.default_desc(accel))
    dev = rt.DeviceRays.from_numpy(scenes.pinhole_rays(64, 48, origin=(0, 0, -3.0)))
    for thr, units in ((0, 0), (rt.RAY_PATH_OFF, 2)):
        for p in (rt.RT_PARAM_RAY_CLUSTERS_CLOSEST, rt.RT_PARAM_RAY_CLUSTERS_OCCLUDED):
            sc.set_param(p, thr)
        sc.set_timing(True)
        for _ in range(2):
            sc.trace_closest(dev)
            sc.trace_occluded(dev)
        for mode in (rt.RT_CLOSEST_PRIMARY, 2):
            ms, n = sc.kernel_time(mode)
            unit, nu = sc.kernel_time(mode + rt.RT_TIME_UNIT)
            ray, nr = sc.kernel_time(mode + rt.RT_TIME_PER_RAY)
            assert (n, nu, nr) == (2, units, 2)
            assert (unit > 0) == (units > 0) and ray > 0 and unit + ray <= ms * 1.001
        sc.set_timing(False)
    sc.close()
