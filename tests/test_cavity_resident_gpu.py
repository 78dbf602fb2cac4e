"""Batches and served launches of a cube with an empty cavity on either side of what the GPU holds at 8 lanes per ray
(6 blocks per CU, where other cubes' kernels have 7): images and counts equal the single renders'."""
import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [7, 8, 9])
def test_cavity_views_equal_their_singles(device, count):
    rng = np.random.default_rng(6)
    vals = (1e-5 * np.exp(rng.standard_normal((40, 44, 48)))).astype(np.float32)
    vals[10:30, 12:33, 9:35] = 0
    vol = capi.Volume.upload(device, vals, (2.0, -8.0, -8.0), (0.35, 0.36, 0.4))
    pos = rng.uniform(-16, 16, (count, 3))
    views = [capi.make_view(100, 60, 50.0, 40.0, tuple(map(float, p)), (10.0, 0.0, 0.0), 40.0, 170) for p in pos]
    want = [vol.render(v) for v in views]
    batch = capi.Batch.exact(vol, views)
    batch.launch()
    batch.wait()
    counts = batch.samples()
    srv = capi.Server(device, memory_budget=1 << 30, max_batch=16, max_inflight=1, batch_window_ms=50.0)
    index = srv.add_volume(vol)
    ids = [srv.submit(index, v) for v in views]
    for k, (img, st) in enumerate(want):
        status, served, _ = srv.wait(ids[k], 20000)
        assert status == capi.OK and counts[k] == st.samples_in_cube
        assert np.array_equal(batch.image(k).view(np.uint32), img.view(np.uint32))
        assert np.array_equal(served.view(np.uint32), img.view(np.uint32))
    assert any(img.any() for img, _ in want)
    srv.destroy()
    batch.free()
    vol.free()
