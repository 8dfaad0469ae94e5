"""Many steps per launch on 1D and small grids against one step per launch
(CH_TB_STEPS=1), bit for bit: each block shape at its smallest and largest grid,
every mobility rule, and step counts on both sides of the launch's depth (32
steps for 1D tiles)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = dict(free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=4, dt=1e-4)
CASES = {
    "landau_euler": dict(integrator="euler", dt=0.004),
    "landau_em_constant": dict(integrator="euler_mobility", dt=0.004, dx=0.9),
    "landau_em_regularised": dict(integrator="euler_mobility", mobility="regularised", rho_min=0.5, dt=1e-3),
    "wertheim_em_linear": dict(integrator="euler_mobility", mobility="linear", rho_ref=0.05, **W),
    "wertheim_em_free_energy": dict(integrator="euler_mobility", mobility="free_energy", **W),
}
GRIDS = [(1, 4), (1, 64), (1, 128), (1, 256), (1, 512), (1, 1024), (1, 2048), (1, 8192),
         (2, 4), (2, 8), (2, 16), (2, 32), (2, 64), (3, 4), (3, 8), (3, 16)]


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("dims,N", GRIDS)
def test_resident_equals_single_steps(ch, ctx, monkeypatch, dims, N, case, precision):
    from cahn_hilliard_amd.init import initial_density
    print(f"case {case} {dims}D N={N} {precision}", flush=True)
    rho = initial_density(dims, N, 0.3 if "landau" in case else 0.05, 0.05, 0, 5 + N)
    got = []
    for tb in ("1", None):
        if tb:
            monkeypatch.setenv("CH_TB_STEPS", tb)
        else:
            monkeypatch.delenv("CH_TB_STEPS")
        s = ch.System(ctx, ch.make_desc(dims=dims, N=N, precision=precision, k=1.0, **CASES[case]))
        assert s.steps_per_launch == 1 if tb else s.steps_per_launch >= 32
        out = []
        for n in (1, 31, 33, 70):
            s.upload(rho)
            s.evolve(n)
            out.append(s.download())
        got.append(out)
        s.close()
    for a, b in zip(*got):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
