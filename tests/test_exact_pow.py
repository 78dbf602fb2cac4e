"""The exact CMEM renders' square root and power (exact_math.h), checked on the CPU; their use in the renders is
compared with the model's own samples, bit for bit, in test_cmem_zones_gpu.py."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pow") / "exact_pow_check")
    subprocess.run(["g++", "-O2", "-std=c++20", "-mfma", "-ffp-contract=off", os.path.join(HERE, "cpu", "exact_pow_check.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("args", [["sqrt", "0"], ["sqrt", "-96"], ["sqrt", "124"], ["pow", "1"], ["pow", "2"]])
def test_within_the_stated_error(exe, args):
    r = subprocess.run([exe] + args, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
