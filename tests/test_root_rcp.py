"""The correctly rounded float root and reciprocal of the device code
(sqrt_rn_f32, rcp_rn in openabl_amd/csrc/abl_device.hpp): a C restatement that
starts from any value within one ulp of the true root or reciprocal (what the
instructions give) against the IEEE operations.  No bound: every result is
equal."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not available")
def test_root_and_reciprocal_are_correctly_rounded(tmp_path):
    exe = str(tmp_path / "root_rcp_check")
    subprocess.run(["gcc", "-O2", "-std=c99", "-ffp-contract=off",
                    os.path.join(HERE, "host", "root_rcp_check.c"), "-o", exe, "-lm"], check=True)
    r = subprocess.run([exe, "500000"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
