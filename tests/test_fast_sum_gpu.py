"""A fast ray's total is its samples' sum rounded once. In a cube of one value v every sample is v, so a pixel of c
samples has to be ((RN(c v) w) K) in FP32, bit for bit: for single renders and batches, every number of
lanes per ray and of samples in flight, cubes without and with negative values (theirs in a corner that
no ray of the views meets)."""
import math

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu
K = np.float32((1.0 * (1000 * 100 * 6378.1) / (4 / math.pi)) / 10000)
VALUE = np.float32(1.2345678e-05)


def check(img, view, where):
    w = np.float32(float(np.float32(view.ray_length)) / view.samples)
    c = np.rint(img.astype(np.float64) / (float(VALUE) * float(w) * float(K)))
    want = ((c * float(VALUE)).astype(np.float32) * w) * K  # c v is exact in FP64
    assert c.max() >= 2, where
    assert np.array_equal(img.view(np.uint32), want.astype(np.float32).view(np.uint32)), (where, int((img != want).sum()), img.size)


@pytest.mark.parametrize("negative", [False, True])
def test_a_constant_cube_sums_to_the_nearest_float(device, negative):
    vals = np.full((20, 20, 20), VALUE, np.float32)
    if negative:
        vals[0, 0, 0] = -VALUE
    vol = capi.Volume.upload(device, vals, (2.0, -5.0, -5.0), (0.5, 0.5, 0.5))
    views = [capi.make_view(w, h, 20.0, 15.0, pos, (6.5, 0.0, 0.0), 40.0, n, capi.SEM_EXTENDED, capi.MATH_FAST)
             for (w, h) in ((33, 21), (200, 120), (451, 347)) for n in (33, 200, 611, 3001) for pos in ((6.5, -14.0, 0.5), (6.0, -13.0, -3.0))]
    for k, v in enumerate(views):
        check(vol.render(v)[0], v, ("single", k))
    batch = capi.Batch(vol, views)
    for t in (None, (8, 8, 1, 4), (8, 8, 1, 1), (8, 4, 2, 4), (4, 8, 2, 1), (4, 4, 4, 4), (4, 4, 4, 1)):
        batch.set_tuning(capi.Tuning(*t) if t else None)
        batch.launch()
        batch.wait()
        for k, v in enumerate(views):
            check(batch.image(k), v, (t, k))
    batch.free()
    vol.free()
