"""Double-precision functions of the evaluation kernels on the device against 80-bit arithmetic on
the host (tests/capi/math_device.cpp): each as exact as the library function or the IEEE operation
that it stands for."""
import os
import subprocess

import pytest

from stormm_amd import build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("function", ["exp", "log", "rsqrt", "tanh", "born_radius", "bond",
                                      "angle"])
def test_error(function):
    exe = os.path.join(build.CAPI_BIN, "math_device")
    if not os.path.exists(exe):
        build.build_capi_programs()
    out = subprocess.run([exe, function], capture_output=True, text=True, timeout=100)
    print(out.stdout)
    assert out.returncode == 0
    assert "math ok" in out.stdout
