"""tests/cpp/host_arithmetic.cpp, built for the host and loaded."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def load(folder):
    from lmdeploy_amd import build
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("hipcc not available")
    out = os.path.join(str(folder), "host_arithmetic.so")
    r = subprocess.run([build._hipcc(), "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-shared", "-fPIC",
                        os.path.join(HERE, "cpp", "host_arithmetic.cpp"), "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return ctypes.CDLL(out)
