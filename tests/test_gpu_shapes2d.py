"""The 2D step's defaults by size, model and mobility, bit for bit against one step
per launch on 64 x 64 regions (CH_WAVE_CFG=4), and the 64 x 40 regions' reverse
sweep against the 64 x 64 ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = dict(free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=4, dt=1e-4)
CASES = {
    "landau_euler": dict(integrator="euler", dt=0.004),
    "landau_em_regularised": dict(integrator="euler_mobility", mobility="regularised", rho_min=0.5, dt=1e-3),
    "wertheim_euler": dict(integrator="euler", **W),
    "wertheim_em_free_energy": dict(integrator="euler_mobility", mobility="free_energy", **W),
}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


def start(case, N):
    from cahn_hilliard_amd.init import initial_density
    return initial_density(2, N, 0.3 if "landau" in case else 0.05, 0.05, 0, 5 + N)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("N", [128, 256, 512, 1024, 2048])
def test_default_shape_equals_single_steps(ch, ctx, monkeypatch, N, case, precision):
    print(f"case {case} N={N} {precision}", flush=True)
    rho, got = start(case, N), []
    for pinned in (False, True):
        if pinned:
            monkeypatch.setenv("CH_WAVE_CFG", "4")
            monkeypatch.setenv("CH_TB_STEPS", "1")
        s = ch.System(ctx, ch.make_desc(dims=2, N=N, precision=precision, k=1.0, **CASES[case]))
        s.upload(rho)
        s.evolve(15)
        s.evolve(8)
        got.append(s.download())
        s.close()
    assert np.all(np.isfinite(got[0])) and np.array_equal(*got)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", ["landau_euler", "wertheim_euler"])
@pytest.mark.parametrize("N,ckpt", [(128, 0), (128, 4), (256, 16)])
def test_region_40_reverse_mode(ch, ctx, monkeypatch, N, ckpt, case, precision):
    """The cells' arithmetic does not depend on the region: dL/dpsi0 bit for bit.  The
    parameter gradients of an FP64 system are sums over regions: n = 23 N^2 terms in
    another order, within n^1/2 ulp of the sum of magnitudes, taken 1e-9 relative (an
    FP32 system's threads sum in FP32; test_gpu_adjoint.py compares those with FP64)."""
    print(f"case {case} N={N} ckpt={ckpt} {precision}", flush=True)
    got = []
    for cfg in ("9", "4"):
        monkeypatch.setenv("CH_ADJ_CFG", cfg)
        s = ch.System(ctx, ch.make_desc(dims=2, N=N, precision=precision, k=1.0, **CASES[case]))
        s.upload(start(case, N))
        s.record(23, ckpt)
        got.append((s.download(), *s.adjoint(np.cos(np.arange(N * N)))))
        s.close()
    for a, b in zip(got[0][:2], got[1][:2]):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
    if precision == "fp64":
        assert np.allclose(got[0][2], got[1][2], rtol=1e-9, atol=0)
