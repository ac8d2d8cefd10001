"""Hyperbolic tangent of the network objective on the GPU against the library's
(tests/cpp/tanh_device_test.hip)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "tanh_device_test")


def test_no_further_off_than_the_library():
    p = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout + p.stderr
