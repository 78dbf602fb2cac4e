"""Exact renders of cubes without negative values (zeros among them, as in an empty cavity) and of nearest
sampling: bit for bit against the oracle on both sides of the rule that picks their kernels -- zeros
of either sign, subnormal values, spacings without the FMA division, an origin at 0, signed cubes --
through single renders, an exact batch and accumulation, and the fast form of the same cubes."""
import os

import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu
NT = min(16, os.cpu_count() or 1)
SHAPE = (37, 30, 41)  # nz, ny, nx


def field(kind, rng):
    v = (1e-5 * np.exp(rng.standard_normal(SHAPE))).astype(np.float32)
    if kind == "cavity":
        z, y, x = np.ogrid[:SHAPE[0], :SHAPE[1], :SHAPE[2]]
        v[(x - 20) ** 2 + (y - 15) ** 2 + (z - 18) ** 2 < 120] = 0
    elif kind == "scattered":
        v[rng.random(SHAPE) < 0.4] = 0
    elif kind == "empty":
        v[:] = 0
    elif kind == "minus_zero":
        v[rng.random(SHAPE) < 0.2] = -0.0
    elif kind == "tiny":
        v[rng.random(SHAPE) < 0.3] = 0
        v[rng.random(SHAPE) < 0.3] *= np.float32(1e-36)
    elif kind == "signed":
        v[rng.random(SHAPE) < 0.002] *= -1
    return v


def oracle_image(O, vals, org, spc, interp, v, sem, init=None):
    ov = O.make_view(v.width, v.height, v.fov_w, v.fov_h, list(v.position), list(v.aim), v.ray_length, v.samples)
    cube = O.OracleCube(vals, org, spc, interp)
    return O.render_f32(cube, ov, sem, nthreads=NT, init=init)


@pytest.mark.parametrize("interp", [capi.INTERP_TRILINEAR, capi.INTERP_NEAREST])
@pytest.mark.parametrize("kind", ["positive", "cavity", "scattered", "empty", "minus_zero", "tiny", "signed"])
@pytest.mark.parametrize("spacing,centred", [(0.4, False), (0.12, False), (0.4, True)])
def test_bitwise(device, oracle, interp, kind, spacing, centred):
    rng = np.random.default_rng(11)
    vals = field(kind, rng)
    org = tuple(0.0 if centred else 8.0 * (k == 0) - 0.5 * spacing * (n - 1) for k, n in enumerate(SHAPE[::-1]))
    mid = [o + 0.5 * spacing * (n - 1) for o, n in zip(org, SHAPE[::-1])]
    vol = capi.Volume.upload(device, vals, org, (spacing,) * 3, interp)
    views = []
    # one image of each lanes-per-ray class, and a camera inside the cube under the reference's semantics
    for (w, h), n, sem in [((61, 43), 90, capi.SEM_EXTENDED), ((150, 101), 33, capi.SEM_EXTENDED), ((301, 173), 64, capi.SEM_EXTENDED),
                           ((320, 200), 51, capi.SEM_REFERENCE)]:
        pos = (mid[0] + 0.7, mid[1] - 1.1, mid[2] + 0.9) if sem == capi.SEM_REFERENCE else (mid[0] - 3.0, mid[1] - 14.0, mid[2] + 5.0)
        views.append(capi.make_view(w, h, 40.0, 30.0, pos, tuple(mid), 30.0, n, sem))
    refs = [oracle_image(oracle, vals, org, (spacing,) * 3, interp, v, v.semantics) for v in views]
    for v, (ref, cnt) in zip(views, refs):
        img, st = vol.render(v)
        assert st.samples_in_cube == cnt and np.array_equal(img.view(np.uint32), ref.view(np.uint32)), (v.width, kind)
    batch = capi.Batch.exact(vol, views)
    batch.launch()
    batch.wait()
    for k, (ref, cnt) in enumerate(refs):
        assert np.array_equal(batch.image(k).view(np.uint32), ref.view(np.uint32))
    assert batch.samples() == [cnt for _, cnt in refs]
    batch.free()
    v = views[1]
    v.flags = capi.RENDER_ACCUMULATE
    init = rng.random((v.height, v.width)).astype(np.float32)
    img, _ = vol.render(v, init=init)
    ref, _ = oracle_image(oracle, vals, org, (spacing,) * 3, interp, v, v.semantics, init=init)
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
    vol.free()


@pytest.mark.parametrize("interp", [capi.INTERP_TRILINEAR, capi.INTERP_NEAREST])
@pytest.mark.parametrize("kind", ["positive", "cavity", "scattered", "minus_zero", "tiny", "signed"])
def test_point_samples_bitwise(device, oracle, interp, kind):
    rng = np.random.default_rng(3)
    vals = field(kind, rng)
    org, spacing = (-3.0, 0.0, 2.0), (0.25, 0.3, 0.12)
    hi = np.array([n - 1 for n in SHAPE[::-1]])
    idx = rng.uniform(-0.5, 1.0, (3000, 3)) * (hi + 0.5)
    idx[:1500] = np.floor(idx[:1500] * 2) / 2  # grid points and midpoints, faces among them
    xyz = (np.array(org) + idx * np.array(spacing)).astype(np.float32)
    vol = capi.Volume.upload(device, vals, org, spacing, interp)
    got = vol.sample(xyz)
    vol.free()
    cube = oracle.OracleCube(vals, org, spacing, interp)
    want = np.array([cube.sample(float(x), float(y), float(z)) for x, y, z in xyz], np.float32)
    assert (want >= 0).any() and (want == -1).any()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("spread", [3.0, 40.0])  # BF16 records as F16 values with one scale, and as BF16
def test_bf16_storage_is_bf16(device, spread):
    rng = np.random.default_rng(4)
    vals = np.exp(rng.uniform(-spread, 0, SHAPE)).astype(np.float32)
    near = (vals.view(np.uint32) + 0x7FFF + (vals.view(np.uint32) >> 16 & 1)) & np.uint32(0xFFFF0000)  # rounded to BF16
    org, spacing = (2.0, -7.0, -6.0), (0.4, 0.4, 0.4)
    v = capi.make_view(97, 61, 40.0, 30.0, (5.0, -20.0, 6.0), (10.0, 0.0, 0.0), 40.0, 300, math=capi.MATH_FAST)
    stored = capi.Volume.upload(device, vals, org, spacing, dtype=capi.DTYPE_BF16)
    rounded = capi.Volume.upload(device, near.view(np.float32), org, spacing)
    a, _ = stored.render(v)
    b = rounded.render_f64(v)
    stored.free()
    rounded.free()
    assert b.any() and np.linalg.norm(a - b) <= 1e-6 * np.linalg.norm(b)
