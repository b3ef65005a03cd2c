"""Adjoint of the particle ladder where its sums run in several a-strips in the
precisions that do not split K (512 tiles of 128 x 128 a strip), off the
multiples of 64 that the packed operands are padded to, in one a-batch and in
several (whose last sum runs over the columns past the batch): every precision
against the FP64 transformation of one a-batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,naux,budget_mb", [(1, 171, 600, 0), (2, 171, 1250, 0), (1, 131, 2500, 1300)])
def test_strips_in_every_precision(o, v, naux, budget_mb, monkeypatch):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system

    eps, B = make_system(o, v, naux, seed=v, sigma=0.01)
    rng = np.random.default_rng(v)
    nov = o * v
    t1, l1 = 0.05 * rng.standard_normal(nov), rng.standard_normal(nov)
    t2, l2 = 0.05 * rng.standard_normal(nov * (nov + 1) // 2), rng.standard_normal(nov * (nov + 1) // 2)
    a_rows = v  # a rows of the first batch, as the budget bounds Y[(a,c),(b,d)]
    if budget_mb:
        a_rows = int(budget_mb * 1e6 / (8.0 * v**3))
        assert 0 < a_rows < v
    assert naux * a_rows * v / 128**2 >= 2 * 512
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(t1, t2)
        ref = c.lhtr(l1, l2, d.FP64, convention="natural")
    if budget_mb:
        monkeypatch.setenv("CCGPU_LADDER_BUDGET_MB", str(budget_mb))
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(t1, t2)
        # rounding of the operands: none, 2^-16 of each (bf16 hi + lo), 2^-24; sums of up to v^2 terms in FP32
        for prec, tol in ((d.FP64, 1e-12), (d.MIXED, 1e-4), (d.FP32, 1e-5)):
            got = c.lhtr(l1, l2, prec, convention="natural")
            err = [np.linalg.norm(g - r) / np.linalg.norm(r) for g, r in zip(got, ref)]
            print(f"adjoint strips o={o} v={v} naux={naux} precision={prec}: {err[0]:.1e} {err[1]:.1e}", flush=True)
            assert max(err) <= tol
