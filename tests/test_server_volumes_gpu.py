"""Registering volumes with a server: what the budget is charged for."""
import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


def test_models_cost_no_budget(device):
    vols = [capi.Volume.cmem(device, capi.cmem_init(capi.cmem_params(density=d))) for d in (5.0, 6.0, 7.0)]
    view = capi.make_view(60, 40, 26.5, 15.5, (0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 60.0, 90)
    srv = capi.Server(device, memory_budget=2 * 60 * 40 * 4, max_batch=4, max_inflight=1)
    try:
        index = [srv.add_volume(v) for v in vols]
        ids = [srv.submit(i, view) for i in index]
        for rid, vol in zip(ids, vols):
            status, img, _ = srv.wait(rid, 20000)
            assert status == capi.OK
            assert np.array_equal(img.view(np.uint32), vol.render(view)[0].view(np.uint32))
    finally:
        srv.destroy()
        for v in vols:
            v.free()


def test_registering_does_not_wait_for_the_device_stream(device):
    """With a long queue of renders on the device's stream, volumes whose making has finished are registered, and
    requests over them served, before the queue ends."""
    rng = np.random.default_rng(2)
    cube = capi.Volume.upload(device, (1e-5 * np.exp(rng.standard_normal((20, 22, 24)))).astype(np.float32), (2.0, -5.0, -4.5), (0.5,) * 3)
    model = capi.Volume.cmem(device, capi.cmem_init())
    image = capi.Image(device, 576, 336)
    long = capi.make_view(576, 336, 26.5, 15.5, (0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 80.0, 8000)
    device.synchronize()

    def queue():
        t = capi.clock_s()
        for _ in range(30):
            capi.render_async(model, long, image)
        return t

    srv = capi.Server(device, memory_budget=1 << 30, max_batch=4, max_inflight=1, reserve_pixels=4096)
    try:
        t = queue()
        device.synchronize()
        whole = capi.clock_s() - t  # about 0.13 s
        assert whole > 0.05
        t = queue()
        srv.add_volume(cube)
        srv.add_volume(model)
        registered = capi.clock_s() - t
        device.synchronize()
        total = capi.clock_s() - t
        assert registered < 0.5 * total, (registered, total)
    finally:
        srv.destroy()
        image.free()
        model.free()
        cube.free()


def test_a_model_made_behind_other_work_is_served_whole(device):
    other = capi.Volume.cmem(device, capi.cmem_init())
    image = capi.Image(device, 576, 336)
    long = capi.make_view(576, 336, 26.5, 15.5, (0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 80.0, 2000)
    views = [capi.make_view(190, 120, 26.5, 15.5, (0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 60.0, 90, capi.SEM_EXTENDED, m)
             for m in (capi.MATH_EXACT, capi.MATH_FAST)]
    srv = capi.Server(device, memory_budget=1 << 30, max_batch=4, max_inflight=2)
    models = []
    try:
        for density in (5.0, 9.0, 14.0):
            for _ in range(10):
                capi.render_async(other, long, image)
            models.append(capi.Volume.cmem(device, capi.cmem_init(capi.cmem_params(density=density))))
            index = srv.add_volume(models[-1])
            ids = [srv.submit(index, v) for v in views]
            got = [srv.wait(i, 20000) for i in ids]
            for (status, img, _), v in zip(got, views):
                assert status == capi.OK
                assert np.array_equal(img.view(np.uint32), models[-1].render(v)[0].view(np.uint32))
    finally:
        srv.destroy()
        image.free()
        for m in models + [other]:
            m.free()



def test_signed_views_of_every_lanes_class_in_one_launch(device):
    """A signed cube's views take 4, 2 or 1 lanes per ray by their own rays and samples (20,000 rays; 150,000 and 64 n^2
    rays): served together, each equals its single render."""
    rng = np.random.default_rng(4)
    vals = (1e-5 * np.exp(rng.standard_normal((30, 32, 34)))).astype(np.float32)
    vals[10:14, 9:13, 11:16] *= -1
    vol = capi.Volume.upload(device, vals, (2.0, -8.0, -7.0), (0.5, 0.5, 0.45))
    views = [capi.make_view(w, h, 50.0, 40.0, (5.0, -18.0, 6.0), (10.0, 0.0, 0.0), 40.0, n, capi.SEM_EXTENDED, capi.MATH_FAST)
             for w, h, n in ((200, 100, 60), (201, 100, 17), (499, 300, 20), (500, 300, 48), (500, 300, 49), (500, 400, 55), (500, 400, 300), (40, 30, 300))]
    want = [vol.render(v)[0] for v in views]
    srv = capi.Server(device, memory_budget=1 << 30, max_batch=8, max_inflight=1, batch_window_ms=50.0)
    try:
        index = srv.add_volume(vol)
        ids = [srv.submit(index, v) for v in views]
        for k, rid in enumerate(ids):
            status, img, _ = srv.wait(rid, 20000)
            assert status == capi.OK and want[k].any()
            assert np.array_equal(img.view(np.uint32), want[k].view(np.uint32)), k
    finally:
        srv.destroy()
        vol.free()
