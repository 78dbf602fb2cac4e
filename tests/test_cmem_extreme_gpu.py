"""CMEM renders equal the model evaluated in full for parameters whose surfaces leave FP32's range somewhere, exact
views bit for bit, and fast views asked by the zone bounds the fast form in full."""
import ctypes as C

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu
PARAMS = [dict(ay_bs=12.0, az_bs=3.0), dict(ay_bs=40.0, az_bs=40.0), dict(ay_bs=-12.0, az_bs=-12.0), dict(ay_bs=3.0, az_bs=-20.0),
          dict(density=10000.0), dict(v=[3000, 0, 0], density=500.0), dict(v=[1200, 0, 0], density=150.0), dict(p1=2000), dict(p1=-2000),
          dict(p3=60), dict(p3=-60), dict(p3=300, p2=0), dict(p0=0.0, p1=-300), dict(bs=1e10), dict(bs=1e-12), dict(p2=1000)]
POSES = [((0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 70.0), ((3.0, 2.0, 15.0), (8.0, 0.0, 0.0), 70.0), ((-30.0, 4.0, 3.0), (10.0, 0.0, 0.0), 70.0),
         ((25.0, -1.0, 2.0), (-5.0, 0.0, 0.0), 70.0), ((200.0, -100.0, 50.0), (0.0, 0.0, 0.0), 600.0), ((2000.0, 500.0, 300.0), (0.0, 0.0, 0.0), 6000.0)]


@pytest.mark.parametrize("params", PARAMS)
def test_renders_equal_the_full_model(device, params):
    vol = capi.Volume.cmem(device, capi.cmem_init(capi.cmem_params(**params)))
    w, h, n = 101, 99, 190  # few enough rays for a single fast view to take the model in full
    L = capi.lib()
    xyz = np.empty((h * w * n, 3), np.float32)
    for pos, aim, length in POSES:
        v = capi.make_view(w, h, 70.0, 50.0, pos, aim, length, n)
        capi.check(L.birp_space_points(device.h, C.byref(v), 0, h, capi.fptr(xyz)), "points")
        vals = vol.sample(xyz)
        want = np.zeros((h, w), np.float32)
        capi.check(L.birp_space_integrate(device.h, C.byref(v), 0, h, capi.fptr(vals), capi.fptr(want)), "integrate")
        got = vol.render(v)[0]
        assert np.array_equal(got.view(np.uint32)[~np.isnan(want)], want.view(np.uint32)[~np.isnan(want)]), pos
        assert np.array_equal(np.isnan(got), np.isnan(want)), pos
        f = capi.make_view(w, h, 70.0, 50.0, pos, aim, length, n, capi.SEM_EXTENDED, capi.MATH_FAST)
        full = vol.render(f)[0]
        batch = capi.Batch(vol, [f])
        batch.set_tuning(capi.Tuning(4, 4, 4, 1))
        batch.launch()
        batch.wait()
        zoned = batch.image(0)
        batch.free()
        assert np.array_equal(np.isnan(full), np.isnan(zoned)) and np.array_equal(full[~np.isnan(full)], zoned[~np.isnan(full)]), pos
    vol.free()
