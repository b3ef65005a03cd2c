"""(T) of a context whose amplitudes were replaced after a first (T): by
set_amplitudes, by the MP2 guess and by a restart file.  The packed layouts of
the amplitudes are kept from call to call, so they must follow; the same
kernels on the same values give the energies of a fresh context."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["launch", "persistent"])
@pytest.mark.parametrize("precision", [0, 1])
def test_pt_follows_the_amplitudes(precision, path, monkeypatch, tmp_path):
    import dalton_amd as d
    from dalton_amd.synthetic import make_system

    monkeypatch.setenv("CCGPU_PT_PATH", path)
    o, v, naux = 3, 21, 40
    eps, B = make_system(o, v, naux, seed=21, sigma=0.01)
    rng = np.random.default_rng(21)
    sets = [(0.05 * rng.standard_normal(o * v), 0.05 * rng.standard_normal(o * v * (o * v + 1) // 2))
            for _ in range(2)]
    ref = []
    for t1, t2 in sets:
        with d.CCContext(eps, B, o) as c:
            c.set_amplitudes(t1, t2)
            ref.append(c.pt(precision))
            c.save_amplitudes(str(tmp_path / f"R0_{len(ref)}"))
    with d.CCContext(eps, B, o) as c:
        c.guess()
        ref.append(c.pt(precision))
    print(f"(T) after new amplitudes, precision {precision}, {path}", flush=True)
    with d.CCContext(eps, B, o) as c:
        c.set_amplitudes(*sets[0])
        got = [c.pt(precision)]
        c.set_amplitudes(*sets[1])
        got.append(c.pt(precision))
        c.guess()
        got.append(c.pt(precision))
        c.restart_amplitudes(str(tmp_path / "R0_1"))
        got.append(c.pt(precision))
    for (a4, a5), (r4, r5) in zip(got, ref + ref[:1]):
        assert abs(a4 - r4) <= 1e-13 * abs(r4) and abs(a5 - r5) <= 1e-13 * max(abs(r5), abs(r4)), (got, ref)
