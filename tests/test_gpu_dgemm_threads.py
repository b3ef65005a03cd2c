"""DGEMM from several threads at once: the calls share the null stream and its
scratch (the partial sums of a split K, the packed operands, which grow from
shape to shape), and each must get its own product."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_threads_get_their_own_products(precision):
    import dalton_amd as d

    rng = np.random.default_rng(8)
    shapes = [(33, 41, 900), (64, 64, 1500), (120, 17, 2000), (200, 150, 700)]  # K split into several chunks each
    ops = [(rng.standard_normal((m, k)), rng.standard_normal((k, n))) for m, n, k in shapes]
    ref = [d.cc.dgemm("N", "N", 1.0, a, b, precision=precision) for a, b in ops]
    for (a, b), r in zip(ops, ref):
        tol = 1e-12 if precision == 0 else 1e-4
        assert np.linalg.norm(r - a @ b) <= tol * np.linalg.norm(a @ b)
    print(f"dgemm threads, precision {precision}", flush=True)
    bad = []

    def work(t):
        for it in range(20):
            q = (t + it) % len(ops)
            c = d.cc.dgemm("N", "N", 1.0, *ops[q], precision=precision)
            if not np.array_equal(c, ref[q]):
                bad.append((t, it, shapes[q], float(np.abs(c - ref[q]).max())))

    th = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for x in th:
        x.start()
    for x in th:
        x.join()
    assert not bad, bad[:5]
