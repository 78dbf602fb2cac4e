"""CMEM renders of points whose squared distances from the Earth or from the Sun's line underflow: exact views equal
the model evaluated in full at the same points, bit for bit (with the angles that FP32 gives there, NaN
among them, as the reference), and fast views, in full or with the zone bounds, the model's fast form in full."""
import ctypes as C

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(9, 7), (110, 100), (260, 240)])
@pytest.mark.parametrize("pos,length", [((3e-20, -2e-20, 1e-20), 2e-19), ((1e-21, 1e-21, -4e-20), 5e-20), ((2e-19, 3e-19, 0.0), 1e-18),
                                        ((0.0, 0.0, 0.0), 3e-19), ((11.0, 2e-20, -1e-20), 1e-19), ((14.5, -3e-23, 2e-22), 4.0),
                                        ((30.0, 1e-25, 1e-24), 60.0), ((1e-21, 11.0, 1e-22), 8.0)])
def test_underflowing_distances(device, size, pos, length):
    vol = capi.Volume.cmem(device, capi.cmem_init())
    L = capi.lib()
    w, h, n = size[0], size[1], 12
    v = capi.make_view(w, h, 40.0, 30.0, pos, (10.0, 0.0, 0.0), length, n)
    xyz = np.empty((h * w * n, 3), np.float32)
    capi.check(L.birp_space_points(device.h, C.byref(v), 0, h, capi.fptr(xyz)), "points")
    vals = vol.sample(xyz)
    want = np.zeros((h, w), np.float32)
    capi.check(L.birp_space_integrate(device.h, C.byref(v), 0, h, capi.fptr(vals), capi.fptr(want)), "integrate")
    got = vol.render(v)[0]
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))

    def fast(a, b):
        f = capi.make_view(a, b, 40.0, 30.0, pos, (10.0, 0.0, 0.0), length, n, capi.SEM_EXTENDED, capi.MATH_FAST)
        return f, vol.render(f)[0]

    f, full = fast(9, 7)  # so few rays take the model in full
    batch = capi.Batch(vol, [f])
    batch.set_tuning(capi.Tuning(4, 4, 4, 1))
    batch.launch()
    batch.wait()
    zoned = batch.image(0)
    batch.free()
    assert np.array_equal(np.isnan(full), np.isnan(zoned)) and np.array_equal(full[~np.isnan(full)], zoned[~np.isnan(zoned)])
    large = fast(w, h)[1]
    vol.free()
    if np.isfinite(full).all():
        assert np.isfinite(large).all()
