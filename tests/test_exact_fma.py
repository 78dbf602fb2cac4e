"""The exact kernels' divisions, scale and lerps as one multiply and one FMA (exact_math.h): checked on
the CPU against the operations they stand for, and on the GPU at the edges of the rule that picks
them -- a spacing for which the division is not exact, values too small for the scale -- bit for
bit against the oracle."""
import os
import subprocess

import numpy as np
import pytest

from birp_cpp_amd import capi

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fma") / "exact_fma_check")
    subprocess.run(["g++", "-O2", "-std=c++20", "-ffp-contract=off", os.path.join(HERE, "cpu", "exact_fma_check.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("args", [["scale"], ["lerp", "1"], ["lerp", "2"]] + [["div", repr(b)] for b in (30 / 255, 30 / 127, 0.1, 0.25, 7.0)])
def test_fma_forms_equal_the_operations(exe, args):
    r = subprocess.run([exe] + args, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_the_division_form_fails_for_some_spacings(exe):
    # 0.12 is one of them: the upload's check is needed
    assert subprocess.run([exe, "div", "0.12"], capture_output=True).returncode == 1


@pytest.mark.gpu
@pytest.mark.parametrize("spacing,amp", [(0.5, 1e-5), (0.12, 1e-5), (0.5, 1e-32), (0.12, 1e-32)])
@pytest.mark.parametrize("size", [(33, 17), (301, 173), (330, 200)])
def test_exact_renders_either_side_of_the_rule(device, oracle, spacing, amp, size):
    rng = np.random.default_rng(5)
    shape = (37, 41, 44)
    vals = (amp * np.exp(rng.standard_normal(shape))).astype(np.float32)
    org = tuple(10.0 * (k == 0) - 0.5 * spacing * (n - 1) for k, n in enumerate(shape[::-1]))
    vol = capi.Volume.upload(device, vals, org, (spacing,) * 3)
    v = capi.make_view(size[0], size[1], 26.5, 15.5, (3.0, -18.0, 6.0), (10.0, 0.0, 0.0), 44.0, 400)
    img, st = vol.render(v)
    vol.free()
    ov = oracle.make_view(v.width, v.height, v.fov_w, v.fov_h, list(v.position), list(v.aim), v.ray_length, v.samples)
    ref, cnt = oracle.render_f32(oracle.OracleCube(vals, org, (spacing,) * 3), ov, oracle.SEM_EXTENDED, nthreads=min(16, os.cpu_count() or 1))
    assert cnt > 0 and st.samples_in_cube == cnt
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
