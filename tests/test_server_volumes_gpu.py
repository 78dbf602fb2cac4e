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
