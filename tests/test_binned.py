"""The likelihood's bin by one exponential (zeus/binned.hpp) against the
formula with power functions, on the host (tests/cpp/binned_test.hip)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bins_equal_the_power_form():
    exe = os.path.join(ROOT, "tests", "cpp", "bin", "binned_test")
    if not os.path.exists(exe):
        from zeus_amd.build import build
        build()
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
