"""The correctly rounded float root and reciprocal of the device code
(sqrt_rn_f32, rcp_rn in openabl_amd/csrc/abl_device.hpp).  No bound: every
result is equal.

  * CPU: their rounding steps (abl_root_rcp.hpp, compiled by the host's compiler)
    from any value within one ulp of the true root or reciprocal, and zeros,
    infinity and NaN;
  * GPU: the functions themselves, from what the instructions give, for every bit
    pattern of a float (roots: without a sign, but for zero).
"""
import ctypes as C
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
DEVICE = os.path.join(REPO, "oracle", "_build", "libroot_rcp_device.so")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_root_and_reciprocal_are_correctly_rounded(tmp_path):
    exe = str(tmp_path / "root_rcp_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    "-I", os.path.join(REPO, "openabl_amd", "csrc"),
                    os.path.join(HERE, "host", "root_rcp_check.cpp"), "-o", exe, "-lm"], check=True)
    r = subprocess.run([exe, "500000"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_device_root_and_reciprocal_for_every_float():
    print("case root and reciprocal of every float", flush=True)
    if not os.path.exists(DEVICE):
        pytest.skip("libroot_rcp_device.so not built")
    bad = (C.c_ulonglong * 2)()
    assert C.CDLL(DEVICE).root_rcp_check(bad) == 0
    assert list(bad) == [0, 0]
