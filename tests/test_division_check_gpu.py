"""The upload's check of the short division per axis: cubes with a spacing for which it is not exact on one axis, two
or all, and with three different ones, render as the oracle, bit for bit."""
import os

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu
BAD, OK, OTHER = 0.12, 0.5, 30 / 127  # tests/test_exact_fma.py checks which is which


@pytest.mark.parametrize("spc", [(BAD, OK, OK), (OK, BAD, OK), (OK, OK, BAD), (OK, OTHER, BAD), (BAD, BAD, OK), (BAD, BAD, BAD), (OK, OTHER, OK), (OTHER, OK, 0.25)])
@pytest.mark.parametrize("interp", [capi.INTERP_TRILINEAR, capi.INTERP_NEAREST])
def test_one_bad_axis_is_enough(device, oracle, spc, interp):
    rng = np.random.default_rng(8)
    n = [int(9.0 / s) for s in spc]
    vals = (1e-5 * np.exp(rng.standard_normal(n[::-1]))).astype(np.float32)
    org = (5.5, -4.6, -4.4)
    vol = capi.Volume.upload(device, vals, org, spc, interp)
    v = capi.make_view(211, 133, 40.0, 30.0, (3.0, -18.0, 6.0), (10.0, 0.0, 0.0), 40.0, 500)
    img, st = vol.render(v)
    vol.free()
    ov = oracle.make_view(v.width, v.height, v.fov_w, v.fov_h, list(v.position), list(v.aim), v.ray_length, v.samples)
    cube = oracle.OracleCube(vals, org, spc, trilinear=interp == capi.INTERP_TRILINEAR)
    ref, cnt = oracle.render_f32(cube, ov, oracle.SEM_EXTENDED, nthreads=min(16, os.cpu_count() or 1))
    assert cnt > 0 and st.samples_in_cube == cnt
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
