"""Device memory of the left transformation and the multipliers, by a dry run
on a device of given size: if a sequence of calls runs on one size it runs on
every larger one.  The DIIS history is kept or released by what the call still
has to allocate; kept where that does not fit, the call fails although a
smaller device, which releases it, gets through."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

SCRIPT = r"""
import ctypes as C, os, sys
import numpy as np
sys.path.insert(0, {root!r})
from dalton_amd import _lib
L = _lib.lib()
x = _lib.ptr(np.zeros(1))  # host arrays are never touched in a dry run
e, r, it = C.c_double(), C.c_double(), C.c_int()
def run(o, v, naux, mb, iterations, what, prec):
    os.environ["CCGPU_DRYRUN_MB"] = str(mb)
    h = C.c_void_p()
    if L.ccgpu_init(o, v, naux, None, None, 8, C.byref(h)):
        return False
    ok = L.ccgpu_ccsd_guess(h, C.byref(e)) == 0
    for p in iterations:
        ok = ok and L.ccgpu_ccsd_iterate(h, p, C.byref(e), C.byref(r)) == 0
    for p in prec:
        if what == "lhtr":
            ok = ok and L.ccgpu_lhtr(h, p, 1, x, x, x, x) == 0
        elif what == "L0":
            ok = ok and L.ccgpu_lambda_solve(h, p, 1e-8, 5, 4, x, x, C.byref(it), C.byref(r)) == 0
        else:
            ok = ok and L.ccgpu_onedens(h, p, x, x, x) == 0
    L.ccgpu_finalize(h)
    return ok
o, v, naux, lo, hi, step = {case!r}
for iterations in ((0,), (1,), (2,), (1, 0)):
    for what, prec in (("lhtr", (0,)), ("lhtr", (1,)), ("lhtr", (2,)), ("lhtr", (0, 1)), ("L0", (0,)), ("L0", (1,)),
                       ("L0", (2,)), ("onedens", (0,)), ("onedens", (1,))):
        got = [(mb, run(o, v, naux, mb, iterations, what, prec)) for mb in range(lo, hi, step)]
        first = next((mb for mb, ok in got if ok), None)
        print(o, v, iterations, what, prec, "from", first, "MB", flush=True)
        assert first is not None and first > lo
        holes = [mb for mb, ok in got if mb > first and not ok]
        assert not holes, (iterations, what, prec, first, holes)
print("done")
"""


@pytest.mark.parametrize("case", [(32, 256, 1024, 30000, 60000, 250), (24, 400, 800, 35000, 75000, 250),
                                  (64, 512, 2048, 200000, 370000, 2500)])
def test_a_larger_device_is_never_too_small(case):
    r = subprocess.run([sys.executable, "-c", SCRIPT.format(root=ROOT, case=case)],
                       env=dict(os.environ, CCGPU_DRYRUN="1"), capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and "done" in r.stdout, r.stdout + r.stderr
