"""FP64 (T) passes against the oracle where the 128 x 128 tile, its 16-row
parts and the K step of 16 end: v and o one below, at and one above."""
import numpy as np
import pytest

from oracle import ccsd as occ
from oracle import triples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v", [(2, 1), (2, 15), (3, 16), (2, 17), (17, 12), (3, 112), (2, 113), (2, 127), (2, 128), (2, 129)])
def test_pt_fp64_tile_edges(o, v):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system

    eps, B = make_system(o, v, 40, seed=3 * o + v)
    print(f"(T) tiles o={o} v={v}", flush=True)
    rng = np.random.default_rng(v)
    t1 = 0.05 * rng.standard_normal((v, o))
    t2 = 0.05 * rng.standard_normal((v, o, v, o))
    t2 = t2 + t2.transpose(2, 3, 0, 1)
    r4, r5 = triples.pt_energy(eps, B, o, t1, t2)
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(occ.pack_t1(t1), occ.pack_t2(t2))
        e4, e5 = c.pt(0)
    # sums of v^3 terms a triple of both signs: rounding grows with the sum of
    # their sizes, which the energies of random amplitudes stay within 1e3 of
    assert abs(e4 - r4) <= 1e-11 * max(1.0, abs(r4))
    assert abs(e5 - r5) <= 1e-11 * max(1.0, abs(r5))
