"""A CMEM model's zone bounds are made for the first render that asks them: whatever that is, its images equal those
of a model in use, and so do the next ones of every other kind."""
import numpy as np
import pytest

from birp_cpp_amd import capi
from test_zz_no_alloc import hip, via_noalloc

pytestmark = pytest.mark.gpu
E, F = capi.MATH_EXACT, capi.MATH_FAST


def view(w, h, math):
    return capi.make_view(w, h, 26.5, 15.5, (0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 60.0, 90, capi.SEM_EXTENDED, math)


EXACT, SMALL, MIDDLE, LARGE = view(190, 120, E), view(60, 40, F), view(190, 120, F), view(300, 210, F)


def use(device, vol, kind):
    if kind in ("exact", "small", "middle", "large"):
        v = dict(exact=EXACT, small=SMALL, middle=MIDDLE, large=LARGE)[kind]
        return [vol.render(v)[0]]
    if kind in ("batch", "exact batch"):
        batch = capi.Batch(vol, [SMALL, LARGE]) if kind == "batch" else capi.Batch.exact(vol, [EXACT])
        batch.launch_graph()
        batch.wait()
        got = [batch.image(k) for k in range(len(batch.views))]
        batch.free()
        return got
    if kind == "noalloc":
        return via_noalloc(hip(), vol, [SMALL, EXACT, LARGE])
    srv = capi.Server(device, memory_budget=1 << 30, max_batch=4, max_inflight=1)
    index = srv.add_volume(vol)
    got = []
    for views in ([EXACT], [LARGE], [SMALL, MIDDLE]):
        ids = [srv.submit(index, v) for v in views]
        got += [srv.wait(i, 20000)[1] for i in ids]
    srv.destroy()
    return got


KINDS = ["exact", "small", "middle", "large", "batch", "exact batch", "noalloc", "server"]


@pytest.mark.parametrize("first", KINDS)
def test_whatever_comes_first(device, first):
    state = capi.cmem_init(capi.cmem_params(density=8.0))
    used = capi.Volume.cmem(device, state)
    used.render(EXACT)
    device.synchronize()
    order = [first] + [k for k in KINDS if k != first]
    want = {k: use(device, used, k) for k in order}
    used.free()
    other = capi.Volume.cmem(device, capi.cmem_init(capi.cmem_params(density=30.0)))  # another's bounds in the freed memory
    other.render(EXACT)
    other.free()
    vol = capi.Volume.cmem(device, state)
    for k in order:
        for a, b in zip(use(device, vol, k), want[k]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), k
    vol.free()
