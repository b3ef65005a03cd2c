"""(T) launched for groups of triples: a group, its remainder and a strided
slice give the sum of the triples taken one by one, at sizes inside one block
tile, past one, and wide enough for the 256 x 256 mixed tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,naux", [(4, 7, 20), (5, 33, 60), (3, 130, 200), (2, 250, 300)])
@pytest.mark.parametrize("precision", [0, 1])
def test_group_is_the_sum_of_its_triples(o, v, naux, precision):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system

    eps, B = make_system(o, v, naux, seed=o + v, sigma=0.02)
    print(f"(T) groups o={o} v={v} precision={precision}", flush=True)
    with d.CCContext(eps, B, o) as c:
        c.guess()
        t1 = 0.01 * np.random.default_rng(v).standard_normal(c.nt1)
        c.set_amplitudes(t1, c.amplitudes()[1])
        n = o * (o + 1) * (o + 2) // 6 - o
        one = [np.array(c.pt_partial(t, 1, 1, precision)[:2]) for t in range(n)]
        full = np.array(c.pt(precision))
        part = np.array(c.pt_partial(1, 3, 2, precision)[:2])
    # the same per-triple values summed in list order on the host
    scale = max(1e-300, np.abs(one).sum())
    assert np.abs(full - sum(one)).max() <= 1e-14 * scale
    assert np.abs(part - sum(one[1::2][:3])).max() <= 1e-14 * scale
