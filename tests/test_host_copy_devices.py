"""Solutions to host arrays on a machine with several devices: copy_to_host compiled for the host against a
stub of the HIP runtime with two of them (tests/host_copy_check.cpp).  Bytes are compared."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_copy_to_host_across_devices(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "host_copy_check")
    subprocess.run([cxx, "-std=c++17", "-O1", "-x", "c++", "-I" + os.path.join(HERE, "hip_stub"),
                    os.path.join(HERE, "host_copy_check.cpp"), "-o", exe, "-pthread"], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(res.stdout)
    assert res.returncode == 0, res.stdout
