"""Products per left transformation: neither the FP32 nor the split-product
GEMM splits K, so the adjoint ladder gives their strips the same number of
tiles, and both precisions take the same launches (the other products do not
depend on the precision)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,naux", [(2, 91, 290), (2, 171, 300), (1, 171, 600)])
def test_unsplit_precisions_take_the_same_strips(o, v, naux):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system

    eps, B = make_system(o, v, naux, seed=v, sigma=0.01)
    rng = np.random.default_rng(v)
    x1, x2 = rng.standard_normal(o * v), rng.standard_normal(o * v * (o * v + 1) // 2)
    n = {}
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(0.01 * x1, 0.01 * x2)
        for prec, name in ((d.FP32, "k_gemm_f32"), (d.MIXED, "k_gemm_bf16x3")):
            c.lhtr(x1, x2, prec)  # the forward intermediates are in place
            d.cc.profile_start()
            c.lhtr(x1, x2, prec)
            n[prec] = d.cc.profile_stop()["kernels"][name]["count"]
    print(f"o={o} v={v} naux={naux}: {n}", flush=True)
    assert n[d.FP32] == n[d.MIXED]
