"""Cubes around the size from which uploads go through the pinned ring (6 MB; chunks of 4 MB, four in the ring): every value
arrives, and the class of the values is found wherever the one that decides it lies."""
import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(95, 128, 129), (96, 128, 128), (97, 127, 131), (64, 256, 256), (65, 253, 259), (131, 201, 203)])
@pytest.mark.parametrize("interp", [capi.INTERP_NEAREST, capi.INTERP_TRILINEAR])
def test_every_value_arrives(device, shape, interp):
    rng = np.random.default_rng(sum(shape))
    vals = rng.uniform(1.0, 2.0, shape).astype(np.float32)
    if interp == capi.INTERP_TRILINEAR:
        vals.reshape(-1)[-1] = -1.0  # the last value alone makes the cube signed: the linear copy is sampled
    vol = capi.Volume.upload(device, vals, (0.5, 0.5, 0.5), (1.0, 1.0, 1.0), interp)
    nz, ny, nx = shape
    z, y, x = np.meshgrid(np.arange(nz - 1), np.arange(ny - 1), np.arange(nx - 1), indexing="ij")
    at = np.stack([x.ravel(), y.ravel(), z.ravel()], 1).astype(np.float32) + np.float32(0.5)
    got = vol.sample(at).reshape(nz - 1, ny - 1, nx - 1)
    vol.free()
    assert np.array_equal(got, vals[:-1, :-1, :-1])


@pytest.mark.parametrize("where", [0, 3 * (1 << 20) + 3, 4259839 - 1])
def test_class_is_found_in_any_chunk(device, where):
    vals = np.full((65, 256, 256), 1e-5, np.float32)  # 4,259,840 values
    vals.reshape(-1)[where] = np.nan
    with pytest.raises(capi.BirpError) as e:  # 16-bit storage needs finite values
        capi.Volume.upload(device, vals, (0.5, 0.5, 0.5), (0.1, 0.1, 0.1), dtype=capi.DTYPE_BF16)
    assert e.value.status == capi.ERR_UNSUPPORTED
    vals.reshape(-1)[where] = 0.0
    vol = capi.Volume.upload(device, vals, (0.5, 0.5, 0.5), (0.1, 0.1, 0.1), dtype=capi.DTYPE_BF16)
    vol.free()
