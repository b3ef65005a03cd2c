"""BF16x3 products on the 64x64 block tile (what small products take without a
timing run) at its edges, against the 128x128 tile bit for bit and against
the exact split-product bound."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# one element; one short of and past a tile and a K step; several tiles, K of one to many steps
CASES = [("N", "N", 1, 1, 1), ("T", "N", 63, 65, 31), ("N", "T", 64, 64, 64), ("T", "T", 65, 129, 200),
         ("N", "N", 130, 70, 96), ("T", "N", 400, 333, 1025)]

_SCRIPT = r"""
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import dalton_amd as d
for q, (ta, tb, m, n, k) in enumerate(%r):
    rng = np.random.default_rng(q)
    A = rng.standard_normal((k, m) if ta == "T" else (m, k))
    B = rng.standard_normal((n, k) if tb == "T" else (k, n))
    C0 = rng.standard_normal((m, n))
    for beta in (0.0, -1.5):
        print("product", ta, tb, m, n, k, beta, flush=True)
        np.save("%%s_%%d_%%d.npy" %% (sys.argv[2], q, beta != 0.0), d.dgemm(ta, tb, 0.75, A, B, beta, C0, precision=d.MIXED))
""" % (CASES,)


def test_small_tile_matches_128_tile(tmp_path):
    for name, env in (("small", {"CCGPU_BF16X3_TUNE": "0"}), ("t128", {"CCGPU_BF16X3_VARIANT": "0"})):
        r = subprocess.run([sys.executable, "-c", _SCRIPT, ROOT, str(tmp_path / name)], env={**os.environ, **env},
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout[-500:] + r.stderr[-500:]
    for q, (ta, tb, m, n, k) in enumerate(CASES):
        rng = np.random.default_rng(q)
        A = rng.standard_normal((k, m) if ta == "T" else (m, k))
        B = rng.standard_normal((n, k) if tb == "T" else (k, n))
        C0 = rng.standard_normal((m, n))
        opA, opB = A.T if ta == "T" else A, B.T if tb == "T" else B
        for beta in (0.0, -1.5):
            got = np.load(tmp_path / f"small_{q}_{int(beta != 0.0)}.npy")
            assert np.array_equal(got, np.load(tmp_path / f"t128_{q}_{int(beta != 0.0)}.npy")), (q, beta)
            # 2^-15 of the products' magnitudes for hi + lo without lo*lo (2^-8 each side twice, halved by
            # rounding), and the FP32 sum of 3k terms
            bound = 0.75 * (2.0**-15 + 3 * k * 2.0**-24) * (np.abs(opA) @ np.abs(opB)) + 1e-14 * np.abs(C0) + 1e-300
            assert (np.abs(got - (0.75 * opA @ opB + beta * C0)) <= bound).all(), (q, beta)
