"""Point samples either side of 2^18 points, where the kernel stops reading the points through the pinned staging that
renders use too: the samples of a long array equal those of its pieces, bit for bit, with renders in between."""
import numpy as np
import pytest

from birp_cpp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["shell", "cavity", "signed", "nearest", "cmem"])
def test_long_arrays_equal_their_pieces(device, oracle, kind):
    rng = np.random.default_rng(9)
    vals = (1e-5 * np.exp(rng.standard_normal((30, 32, 34)))).astype(np.float32)
    if kind == "cavity":
        vals[8:20, 8:20, 8:20] = 0
    if kind == "signed":
        vals[8:20, 8:20, 8:20] *= -1
    org, spc = (2.0, -8.0, -7.0), (0.5, 0.5, 0.45)
    if kind == "cmem":
        vol = capi.Volume.cmem(device, capi.cmem_init())
    else:
        vol = capi.Volume.upload(device, vals, org, spc, capi.INTERP_NEAREST if kind == "nearest" else capi.INTERP_TRILINEAR)
    view = capi.make_view(301, 173, 40.0, 30.0, (3.0, -18.0, 6.0), (10.0, 0.0, 0.0), 40.0, 60)
    image = vol.render(view)[0]
    n = (1 << 18) + 1
    xyz = (rng.uniform(-1.1, 1.1, (n, 3)) * (9.0, 9.0, 8.0) + (9.0, 0.0, 0.0)).astype(np.float32)
    long = vol.sample(xyz)
    for first, count in ((0, 1), (0, 1000), (5, 70001), (1, 1 << 18), (0, 1 << 18)):
        got = vol.sample(xyz[first:first + count])
        assert np.array_equal(got.view(np.uint32), long[first:first + count].view(np.uint32)), (first, count)
        assert np.array_equal(vol.render(view)[0].view(np.uint32), image.view(np.uint32))
    vol.free()
    if kind != "cmem":
        cube = oracle.OracleCube(vals, org, spc, trilinear=kind != "nearest")
        for k in range(0, n, 2111):
            assert np.float32(cube.sample(*map(float, xyz[k]))) == long[k], k
        assert (long != -1).any() and (long == -1).any()
