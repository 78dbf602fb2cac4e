"""Fast images of cubes without negative values do not depend on the launch: every tuning of a batch (tile, lanes
per ray, samples in flight), the single render and a batch of many more views give the same bits, for
every storage, at image sizes and sample counts off the tiles and the 16-sample groups."""
import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu
TUNINGS = [(8, 8, 1, 4), (16, 4, 1, 1), (8, 4, 2, 4), (4, 8, 2, 2), (2, 16, 2, 1), (4, 4, 4, 4), (8, 2, 4, 2), (2, 8, 4, 1)]


@pytest.mark.parametrize("dtype", [capi.DTYPE_F32, capi.DTYPE_BF16, capi.DTYPE_F16])
@pytest.mark.parametrize("kind", ["shell", "cavity", "wide"])
def test_images_do_not_depend_on_the_tuning(device, dtype, kind):
    rng = np.random.default_rng(7)
    shape = (41, 35, 50)
    vals = (1e-5 * np.exp(0.5 * rng.standard_normal(shape))).astype(np.float32)
    if kind == "cavity":
        vals[10:30, 8:25, 12:40] = 0
    if kind == "wide":  # FP16: a scale per brick
        vals *= np.float32(10.0) ** rng.integers(-14, 14, (1, 1, shape[2])).astype(np.float32)
    vol = capi.Volume.upload(device, vals, (2.0, -8.0, -7.0), (0.4, 0.45, 0.35), dtype=dtype)
    views = [capi.make_view(w, h, 60.0, 45.0, pos, (10.0, 0.0, 0.0), 30.0, n, sem, capi.MATH_FAST)
             for (w, h), n, pos, sem in [((33, 21), 15, (5.0, -14.0, 6.0), capi.SEM_EXTENDED), ((70, 50), 16, (11.0, 1.0, -2.0), capi.SEM_REFERENCE),
                                         ((129, 65), 17, (-3.0, 4.0, 9.0), capi.SEM_EXTENDED), ((64, 64), 203, (5.0, -14.0, 6.0), capi.SEM_EXTENDED),
                                         ((1, 1), 64, (11.0, 1.0, -2.0), capi.SEM_EXTENDED), ((301, 173), 90, (22.0, 9.0, 1.0), capi.SEM_EXTENDED)]]
    want = [vol.render(v)[0] for v in views]
    assert all(np.isfinite(w).all() for w in want) and any((w > 0).any() for w in want)
    batch = capi.Batch(vol, views)
    for t in TUNINGS:
        batch.set_tuning(capi.Tuning(*t))
        batch.launch()
        batch.wait()
        for k, w in enumerate(want):
            assert np.array_equal(batch.image(k).view(np.uint32), w.view(np.uint32)), (t, k)
    batch.free()
    many = capi.Batch(vol, views * 70)
    many.launch()
    many.wait()
    for k in range(len(views) * 66, len(views) * 70):
        assert np.array_equal(many.image(k).view(np.uint32), want[k % len(views)].view(np.uint32))
    many.free()
    f64 = vol.render_f64(views[5]) if dtype == capi.DTYPE_F32 else None
    if f64 is not None:
        assert np.linalg.norm(want[5] - f64) <= 1e-5 * np.linalg.norm(f64)
    vol.free()
