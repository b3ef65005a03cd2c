"""(T) launched for groups of triples, past one group and past one range of
descriptors (4096 triples), none of them a multiple of the group: the whole
list, whose host descriptors are refilled per range, against strided slices
of it and single triples."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("o,v", [(8, 9), (30, 4)])
def test_groups_and_ranges_add_up(o, v, precision):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system

    eps, B = make_system(o, v, 30, seed=o, sigma=0.01)
    rng = np.random.default_rng(o)
    nov = o * v
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(0.05 * rng.standard_normal(nov), 0.05 * rng.standard_normal(nov * (nov + 1) // 2))
        e4, e5, fl, nt = c.pt_partial(0, 10**9, 1, precision)
        print(f"o={o} v={v} precision={precision}: {nt} triples", flush=True)
        assert nt > 64 and nt % 64 and (o != 30 or nt > 4096)
        parts = [c.pt_partial(q, 10**9, 3, precision) for q in range(3)]
        one = [c.pt_partial(q, 1, 1, precision) for q in range(nt - 70, nt)]
        tail = c.pt_partial(nt - 70, 70, 1, precision)
    # sums of the same per-triple values in another order
    s4, s5 = sum(abs(p[0]) for p in parts), sum(abs(p[1]) for p in parts)
    assert abs(sum(p[0] for p in parts) - e4) <= 1e-12 * s4 and abs(sum(p[1] for p in parts) - e5) <= 1e-12 * s5
    assert abs(sum(p[0] for p in one) - tail[0]) <= 1e-12 * sum(abs(p[0]) for p in one)
    assert abs(sum(p[1] for p in one) - tail[1]) <= 1e-12 * sum(abs(p[1]) for p in one)
