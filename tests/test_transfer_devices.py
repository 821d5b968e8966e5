"""elmm_upload and elmm_download of a handle whose device is not the calling
thread's current one, on a stand-in for the HIP runtime (hip_two_devices.cpp):
the slots' events belong to the handle's device, the caller's stays current."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

SCRIPT = """
import ctypes, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the HIP runtime itself
sys.path.insert(0, sys.argv[2])
import numpy as np
from elmm_amd import capi, cases

def device():
    d = ctypes.c_int(-1)
    hip.hipGetDevice(ctypes.byref(d))
    return d.value

n = int(sys.argv[3])
cfg = cases.uniform_config(n, n, n, dx=1.0, dt=0.02, nscalars=1)
case = capi.Case(cfg)
solvers = []
for d in (0, 1):
    hip.hipSetDevice(d)
    solvers.append(capi.Solver(cfg, case))
rng = np.random.default_rng(1)
for d in (0, 1):
    hip.hipSetDevice(d)
    for s in solvers:
        for field in (capi.F_U, capi.F_SCALAR):
            a = rng.standard_normal(capi.ghosted_shape(cfg))
            s.upload(field, a)
            assert device() == d, "upload changed the caller's device"
            assert np.array_equal(s.download(field), a)
            assert device() == d, "download changed the caller's device"
print("ok")
"""


# one task, on the caller's thread; several, on threads of their own
@pytest.mark.parametrize("n", [8, 96])
def test_transfers_of_a_handle_on_another_device(tmp_path, n):
    lib = str(tmp_path / "libhip_two_devices.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    os.path.join(HERE, "hip_two_devices.cpp"), "-o", lib], check=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, lib, os.path.join(os.path.dirname(HERE), "gpu-elmm_amd"), str(n)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
