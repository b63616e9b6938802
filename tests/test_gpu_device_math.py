"""The device kernels' short arithmetic against what it stands for
(tests/csrc/check_device_math.hip, run as a program of its own)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc", "check_device_math")


def test_device_math():
    assert os.path.exists(EXE), "built by legitengine_amd.build"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
