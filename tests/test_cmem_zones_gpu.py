"""The CMEM renders leave the model's surfaces out where their zone bounds name a point's zone: every image has
to equal, bit for bit, the integration of the model evaluated in full at the same points
(birp_space_points, birp_volume_sample, birp_space_integrate), for parameters that move, tilt and
distort the surfaces, from every side, along the axes and far down the tail."""
import ctypes as C

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu

PARAMS = [dict(), dict(p0=1.0, p1=4, p2=6, p3=3, B=3.6, alpha=-1.0), dict(ay_bs=0.9, az_bs=0.5), dict(dipole=0.4, density=20.0),
          dict(dipole=-0.9, b=[3, -2, -18]), dict(v=[800, 0, 0], density=60.0, bs=9.0), dict(v=[250, 0, 0], density=0.5, p3=1),
          dict(p1=-2, ay_bs=-0.3, az_bs=0.2), dict(bs=-5.0)]
POSES = [((0.0, -20.0, 10.0), (10.0, 0.0, 0.0)), ((3.0, 2.0, 15.0), (8.0, 0.0, 0.0)), ((-30.0, 4.0, 3.0), (10.0, 0.0, 0.0)),
         ((25.0, -1.0, 2.0), (-5.0, 0.0, 0.0)), ((0.0, 0.0, 12.0), (10.0, 0.0, 0.0))]


@pytest.mark.parametrize("params", PARAMS)
@pytest.mark.parametrize("pos,aim", POSES)
def test_render_equals_the_full_model(device, params, pos, aim):
    vol = capi.Volume.cmem(device, capi.cmem_init(capi.cmem_params(**params)))
    w, h, n = 57, 35, 190
    v = capi.make_view(w, h, 70.0, 50.0, pos, aim, 70.0, n)
    L = capi.lib()
    xyz = np.empty((h * w * n, 3), np.float32)
    capi.check(L.birp_space_points(device.h, C.byref(v), 0, h, capi.fptr(xyz)), "points")
    vals = vol.sample(xyz)
    want = np.zeros((h, w), np.float32)
    capi.check(L.birp_space_integrate(device.h, C.byref(v), 0, h, capi.fptr(vals), capi.fptr(want)), "integrate")
    got, _ = vol.render(v)
    batch = capi.Batch.exact(vol, [v])
    batch.launch()
    batch.wait()
    other = batch.image(0)
    batch.free()
    vol.free()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(other.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("size", [(40, 30), (150, 100), (280, 200), (330, 210)])
def test_every_lanes_per_ray_class(device, size):
    vol = capi.Volume.cmem(device, capi.cmem_init())
    v = capi.make_view(size[0], size[1], 26.5, 15.5, (1.0, -18.0, 8.0), (10.0, 0.0, 0.0), 60.0, 61)
    single, st = vol.render(v)
    batch = capi.Batch.exact(vol, [v])
    batch.launch()
    batch.wait()
    assert np.array_equal(single.view(np.uint32), batch.image(0).view(np.uint32))
    assert st.samples_in_cube == batch.samples()[0] == size[0] * size[1] * 61
    batch.free()
    vol.free()


@pytest.mark.parametrize("params", PARAMS)
def test_fast_views_of_every_size_equal_the_batch(device, params):
    """A single fast view asks the zone bounds in the way of its size (in full up to 10,000 rays, a trip ahead up
    to 60,000, before each sample above), a launch of many before each sample: with the same lanes
    per ray, which order a ray's sum, the images are the same bits."""
    vol = capi.Volume.cmem(device, capi.cmem_init(capi.cmem_params(**params)))
    views = [capi.make_view(w, h, 70.0, 50.0, pos, aim, 70.0, n, capi.SEM_EXTENDED, capi.MATH_FAST)
             for (pos, aim) in POSES for (w, h, n) in ((1, 1, 2), (33, 21, 67), (100, 100, 41), (101, 100, 66), (240, 250, 30), (241, 250, 31))]
    batch = capi.Batch(vol, views)
    batch.set_tuning(capi.Tuning(4, 4, 4, 1))
    batch.launch()
    batch.wait()
    for k, v in enumerate(views):
        got = vol.render(v)[0]
        assert np.array_equal(got.view(np.uint32), batch.image(k).view(np.uint32)), k
    batch.free()
    vol.free()
