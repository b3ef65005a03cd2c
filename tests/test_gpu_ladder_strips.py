"""Particle ladder and its adjoint at the edges of its tiles (32 and 128 virtual
orbitals, rows of four) and where one a-batch is formed in several a-strips
(v = 90 and 91: three strips, the adjoint two, off every tile and K-step
boundary): residual and left transformation against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,naux", [(1, 31, 40), (2, 32, 40), (5, 33, 40), (6, 36, 40), (2, 90, 300), (3, 91, 290),
                                      (1, 128, 60), (1, 129, 60)])
def test_strips_match_oracle(o, v, naux):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system
    from oracle import ccsd as occ
    from oracle import lhtr as olh

    eps, B = make_system(o, v, naux, seed=v, sigma=0.01)
    sysm = occ.DFSystem(eps, B, o)
    rng = np.random.default_rng(v)
    t1 = 0.05 * rng.standard_normal((v, o))
    t2 = 0.05 * rng.standard_normal((v, o, v, o))
    t2 = t2 + t2.transpose(2, 3, 0, 1)
    p1, p2 = occ.pack_t1(t1), occ.pack_t2(t2)
    l1, l2 = rng.standard_normal(p1.size), rng.standard_normal(p2.size)
    r1, r2 = occ.residual(sysm, t1, t2)
    q1, q2 = olh.left_transform(sysm, p1, p2, l1, l2)
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(p1, p2)
        for prec, tol in ((d.FP64, 1e-12), (d.MIXED, 1e-4)):
            print(f"ladder strips o={o} v={v} precision={prec}", flush=True)
            om1, om2 = c.rhs(p1, p2, prec)
            g1, g2 = c.lhtr(l1, l2, prec, convention="natural")
            for got, ref in ((om1, occ.pack_t1(r1)), (om2, occ.pack_t2(r2)), (g1, q1), (g2, q2)):
                assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), prec
