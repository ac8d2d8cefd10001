"""Hyperbolic tangent (zeus/tanh.hpp) against long double, on the host
(tests/cpp/tanh_test.hip)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tanh_against_long_double():
    exe = os.path.join(ROOT, "tests", "cpp", "bin", "tanh_test")
    if not os.path.exists(exe):
        from zeus_amd.build import build
        build()
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
