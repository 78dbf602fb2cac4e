"""Fast batches of more blocks than one grid may have (2^24 of 256 threads) take several launches: the split on
the CPU, and on the GPU a batch of 2^24 blocks and more against its views' single renders."""
import os
import subprocess

import numpy as np
import pytest

from birp_cpp_amd import capi

HERE = os.path.dirname(os.path.abspath(__file__))


def test_pieces_cover_every_block_once(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "cpu", "fast_pieces_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_a_batch_of_more_blocks_than_a_grid(device):
    # 4 lanes per ray: 64 rays to a block, 4 x 2^22 blocks and those of the small views
    vol = capi.Volume.cmem(device, capi.cmem_init())
    def view(w, h, n):
        return capi.make_view(w, h, 26.5, 15.5, (0.0, -20.0, 10.0), (10.0, 0.0, 0.0), 40.0, n, capi.SEM_EXTENDED, capi.MATH_FAST)
    views = [view(70, 50, 33)] + [view(1 << 14, 1 << 14, 2)] * 4 + [view(41, 33, 60)]
    batch = capi.Batch(vol, views)
    try:
        for launch in (batch.launch, batch.launch_graph):
            launch()
            batch.wait()
            for k in (0, 5):
                want = vol.render(views[k])[0]
                assert want.any() and np.array_equal(batch.image(k).view(np.uint32), want.view(np.uint32)), k
        big = batch.image(1)
        assert np.isfinite(big[::97]).all() and (big[::97] > 0).any()
        assert np.array_equal(batch.image(4).view(np.uint32), big.view(np.uint32))
    finally:
        batch.free()
        vol.free()
