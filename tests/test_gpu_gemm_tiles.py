"""FP64 GEMM at the edges of its 32, 64 and 128 block tiles, of their K steps
(64, 32 and 16) and of the split of K, in every operand order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k): one element, one short of and one past a tile or a K step, long K
# over a small result (many chunks), and shapes wide enough for the 64 and 128 tiles
SIZES = [
    (1, 1, 1), (5, 19, 1), (31, 33, 63), (32, 32, 64), (33, 31, 65), (5, 5, 1805), (21, 170, 4099), (1, 300, 2500),
    (900, 1100, 31), (1000, 1001, 33), (64, 8200, 129), (1700, 1900, 15), (2049, 1663, 17), (1793, 2177, 683),
]


@pytest.mark.parametrize("m,n,k", SIZES)
def test_dgemm_at_tile_edges(m, n, k):
    import dalton_amd as d

    rng = np.random.default_rng(m + 3 * n + 7 * k)
    A, B, C0 = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    ref = -0.75 * (A @ B) + 0.5 * C0
    # each result sums k products and two terms, here and in numpy, every
    # rounding at most eps of the sum of magnitudes
    eps = np.finfo(np.float64).eps
    bound = 2.0 * (k + 4) * eps * (0.75 * (np.abs(A) @ np.abs(B)) + 0.5 * np.abs(C0))
    for ta in "NT":
        for tb in "NT":
            print(f"dgemm {ta}{tb} m={m} n={n} k={k}", flush=True)
            got = d.dgemm(ta, tb, -0.75, A.T if ta == "T" else A, B.T if tb == "T" else B, 0.5, C0)
            assert (np.abs(got - ref) <= bound).all(), (ta, tb)
