"""Templated objectives in a caller's own numbers and in float
(tests/cpp/generic_objectives_test.hip), on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_own_numbers():
    exe = os.path.join(ROOT, "tests", "cpp", "bin", "generic_objectives_test")
    if not os.path.exists(exe):
        from zeus_amd.build import build
        build()
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
