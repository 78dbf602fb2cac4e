"""Exact images wider than 2^24 pixels: the reference divides by the width converted to FP32 (Camera.cpp:148), which
no longer holds every integer there."""
import os

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [(1 << 24) + 1, (1 << 24) + 3])
def test_a_row_of_more_pixels_than_a_float_counts(device, oracle, width):
    rng = np.random.default_rng(3)
    vals = (1e-5 * np.exp(0.5 * rng.standard_normal((18, 20, 22)))).astype(np.float32)
    org, spc = (4.5, -5.0, -4.5), (0.5, 0.5, 0.5)
    pos, aim, fov = (9.0, -14.0, 1.0), (10.0, 0.0, 0.0), (3e-6, 2.0)
    vol = capi.Volume.upload(device, vals, org, spc)
    img, st = vol.render(capi.make_view(width, 1, *fov, pos, aim, 24.0, 3))
    vol.free()
    ov = oracle.make_view(width, 1, *fov, list(pos), list(aim), 24.0, 3)
    ref, cnt = oracle.render_f32(oracle.OracleCube(vals, org, spc), ov, oracle.SEM_EXTENDED, nthreads=min(16, os.cpu_count() or 1))
    assert cnt > width // 4 and st.samples_in_cube == cnt
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
