"""Fast images over 16-bit cubes scale with the cube: values times a power of two give the image times that power,
bit for bit, down to values whose FP16 records' common scale is the smallest normal float."""
import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [capi.DTYPE_BF16, capi.DTYPE_F16])
@pytest.mark.parametrize("power", [-95, -60, 0, 60, 100])
@pytest.mark.parametrize("negative", [False, True])
def test_images_scale_with_the_cube(device, dtype, power, negative):
    rng = np.random.default_rng(12)
    vals = (1e-5 * np.exp(0.4 * rng.standard_normal((20, 22, 24)))).astype(np.float32)
    if negative:
        vals[3, 4, 5] *= -1
    # the largest value in [2^-16, 2^-15): FP16 records' scale 2^-30, times 2^-95 2^-125
    vals *= np.float32(0.75 * 2.0**-15 / np.abs(vals).max())
    views = [capi.make_view(w, h, 60.0, 45.0, pos, (10.0, 0.0, 0.0), length, n, capi.SEM_EXTENDED, capi.MATH_FAST)
             for (w, h), pos, length, n in [((61, 43), (5.0, -14.0, 6.0), 30.0, 700), ((211, 130), (11.0, 1.0, -2.0), 0.5, 90)]]
    images = []
    for p in (0, power):
        vol = capi.Volume.upload(device, vals * np.float32(2.0) ** p, (2.0, -5.0, -4.5), (0.5, 0.45, 0.5), dtype=dtype)
        images.append([vol.render(v)[0] for v in views])
        vol.free()
    for a, b in zip(*images):
        assert (a > 0).any()
        assert np.array_equal((a.astype(np.float64) * 2.0**power).astype(np.float32).view(np.uint32), b.view(np.uint32))
