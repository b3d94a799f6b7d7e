"""The stage kernels' own arithmetic at the values where it can go wrong: zeros,
infinities, NaN, subnormals (tests/cpp/test_device_math.hip)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

BINARY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build", "test_device_math")


def test_against_ieee_arithmetic():
    r = subprocess.run([BINARY], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "PASS" in r.stdout
