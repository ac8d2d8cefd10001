"""The Gaussian as a functor of zeus::Zeus (tests/cpp/functor_gaussian_test.hip)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin",
                   "functor_gaussian_test")


def test_every_start_converges(tmp_path):
    p = subprocess.run([EXE], capture_output=True, text=True, timeout=100, cwd=tmp_path)
    assert p.returncode == 0, p.stdout + p.stderr
