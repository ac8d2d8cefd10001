"""The inverse Hessian as a list of rank-2 pairs with folds (PairMatrix),
against the explicit matrix (tests/cpp/pair_matrix_test.hip)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "pair_matrix_test")


def test_products_across_folds():
    p = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout + p.stderr
