"""A wait of the eigen solver that fails is reported, not taken for the end of its
rounds.  Run in a process that sees no GPU: every launch and the wait then fail,
and nothing is executed."""
import os
import subprocess
import sys

import pytest

from openrcwa_amd import _lib

CALL = """
import ctypes, subprocess, sys
lib = ctypes.CDLL(sys.argv[1])
count = ctypes.c_int(-1)
hip = ctypes.CDLL("libamdhip64.so")
if hip.hipGetDeviceCount(ctypes.byref(count)) == 0 and count.value > 0:
    sys.exit(77)                      # a GPU is visible after all: not to be called
names = subprocess.run(["nm", "-D", "--defined-only", sys.argv[1]], check=True,
                       capture_output=True, text=True).stdout.split()
zgeev = getattr(lib, next(s for s in names if "zgeev_batched" in s))
P, I = ctypes.c_void_p, ctypes.c_int
zgeev.argtypes = [P, I, P, P, P, P, P, P, P, P, I, P, ctypes.c_double, I, ctypes.c_bool, P]
zgeev.restype = I
ws = (P * 3)()
route = (I * 2)(-1, 0)
error = zgeev(None, 200, None, None, None, None, ctypes.addressof(ws), None, None, None, 1, None,
              1e-8, 0, True, ctypes.addressof(route))
print("error", error)
sys.exit(0 if 0 < error < 2000 else 1)
"""


def test_a_failed_wait_is_an_error():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1")
    r = subprocess.run([sys.executable, "-c", CALL, _lib.LIB_PATH], env=env, timeout=60,
                       capture_output=True, text=True)
    if r.returncode == 77:
        pytest.skip("a GPU is visible")
    assert r.returncode == 0, r.stdout + r.stderr
