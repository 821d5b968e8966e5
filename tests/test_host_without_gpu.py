"""Host code of the engine on a stand-in for the HIP runtime
(hip_standin.cpp), without a GPU: transfers of a handle whose device is not
the calling thread's current one, and the autotuner's cache beside settings
fixed by the environment."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from elmm_amd import capi

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, os, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the HIP runtime itself
sys.path.insert(0, sys.argv[2])
import numpy as np
from elmm_amd import capi, cases
"""

TRANSFERS = """
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

TUNED = """
cfg = cases.uniform_config(64, 64, 256, dx=1.0, dt=0.02, nscalars=1, autotune=1)
case = capi.Case(cfg)

def tiles(env):
    if env:
        os.environ["ELMM_SGS_ZCHUNK"] = env
    else:
        os.environ.pop("ELMM_SGS_ZCHUNK", None)
    s = capi.Solver(cfg, case)
    s.init()
    s.step(1, diag=False)
    return s.tiles()["sgs_zchunk"]

got = [tiles(e) for e in sys.argv[3].split(",")]
assert all(g == int(e) if e else g in (13, 16, 26, 32) for g, e in zip(got, sys.argv[3].split(","))), got
print("ok")
"""

# a handle that a static object of the program destroys, as the process ends
AT_EXIT = """
cfg = cases.uniform_config(48, 48, 48, dx=1.0, dt=0.02)
s = capi.Solver(cfg, capi.Case(cfg))
s.upload(capi.F_U, np.zeros(capi.ghosted_shape(cfg)))
owner = ctypes.CDLL(sys.argv[3])
owner.own.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
owner.own(s._h, ctypes.cast(capi._lib.elmm_destroy, ctypes.c_void_p))
s._h = None
print("ok")
"""

OWNER = """
#include <cstdlib>
static void *handle;
static int (*destroy)(void *);
struct Owner {
  ~Owner() {
    if (destroy && destroy(handle)) std::_Exit(4);
  }
};
static Owner owner;
extern "C" void own(void *h, int (*d)(void *)) {
  handle = h;
  destroy = d;
}
"""


def _run(tmp_path, script, arg):
    lib = str(tmp_path / "libhip_standin.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    os.path.join(HERE, "hip_standin.cpp"), "-o", lib], check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + script, lib,
                        os.path.join(os.path.dirname(HERE), "gpu-elmm_amd"), arg],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


# one task, on the caller's thread; several, on threads of their own; no memory
# to be had for pinned slots
@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("n", [8, 96])
def test_transfers_of_a_handle_on_another_device(tmp_path, monkeypatch, n, pinned):
    if not pinned:
        monkeypatch.setenv("STANDIN_NO_PINNED_MEMORY", "1")
    _run(tmp_path, TRANSFERS, str(n))


def test_handle_destroyed_by_a_static_object(tmp_path):
    src, lib = tmp_path / "owner.cpp", tmp_path / "libowner.so"
    src.write_text(OWNER)
    subprocess.run(["g++", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    # loaded before the library's own static objects exist
    _run(tmp_path, "ctypes.CDLL(sys.argv[3])\n" + AT_EXIT, str(lib))


# a chunk fixed after a tuned handle, and before one (whose room for the SGS
# kernel's partials is sized by the chunks that the tuner tries)
@pytest.mark.parametrize("order", [",4", "4,", "40,,4"])
def test_tuned_choices_and_fixed_settings_stay_apart(tmp_path, order):
    _run(tmp_path, TUNED, order)


# the z solve's table of pivots is used where it is the faster solve: not where
# its columns leave a CU few blocks and the grid has many modes, nor beyond a
# CU's LDS (arguments: modes a row, rows, levels)
@pytest.mark.parametrize("modes,used", [((40, 64, 64), 1), ((40, 64, 392), 1), ((40, 64, 400), 0),
                                        ((136, 256, 192), 1), ((136, 256, 200), 0), ((200, 256, 128), 1),
                                        ((200, 256, 136), 0), ((264, 512, 64), 0)])
def test_pivot_table_where_it_is_faster(modes, used):
    wanted = capi.load()._ZN4elmm14z_table_wantedEiii
    wanted.argtypes, wanted.restype = [C.c_int] * 3, C.c_bool
    assert wanted(*modes) == bool(used)
