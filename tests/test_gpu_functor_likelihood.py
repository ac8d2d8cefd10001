"""The binned likelihood as a functor of zeus::Zeus against the built-in
(tests/cpp/functor_likelihood_test.hip)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin",
                   "functor_likelihood_test")


def test_functor_equals_builtin(tmp_path):
    p = subprocess.run([EXE], capture_output=True, text=True, timeout=100, cwd=tmp_path)
    assert p.returncode == 0, p.stdout + p.stderr
