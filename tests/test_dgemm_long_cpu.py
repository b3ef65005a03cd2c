"""Long thin FP64 products whose 32 x 32 tiles do not fit a grid, by the host
checks of a dry run (no memory is allocated, nothing is launched)."""
import os
import subprocess
import sys

from conftest import ROOT

SCRIPT = r"""
import ctypes as C, sys
import numpy as np
sys.path.insert(0, {root!r})
from dalton_amd import _lib
L = _lib.lib()
h = C.c_void_p()
assert L.ccgpu_init(1, 1, 1, None, None, 8, C.byref(h)) == 0
x = _lib.ptr(np.zeros(1))  # host arrays are never touched in a dry run
for big in (536870911, 540000000, 1070000000):
    for small in (1, 16, 33):
        for k in (0, 1, 17, 32, 48):
            for m, n in ((small, big), (big, small)):
                rc = L.ccgpu_dgemm(b"N", b"N", m, n, k, 1.0, x, m, x, max(1, k), 0.0, x, m)
                assert rc == 0, (m, n, k, L.ccgpu_last_error())
rc = L.ccgpu_dgemm(b"N", b"N", 1, 2**31 - 1, 1, 1.0, x, 1, x, 1, 0.0, x, 1)  # past 2^24 tiles of 128
assert rc == 1 and b"too many tiles" in L.ccgpu_last_error()
print("ok")
"""


def test_long_products_are_accepted():
    r = subprocess.run([sys.executable, "-c", SCRIPT.format(root=ROOT)], env=dict(os.environ, CCGPU_DRYRUN="1"),
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
