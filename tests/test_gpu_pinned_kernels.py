"""CH_WAVE_CFG at 2D N = 64 and CH_TILE3D up to 3D N = 16 run the kernels they name,
not the many-step launches of those grids, with the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = dict(integrator="euler_mobility", free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=4, mobility="linear",
         rho_ref=0.05, dt=1e-4)


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("dims,N,env,values,depth", [(2, 64, "CH_WAVE_CFG", "034", 8), (3, 16, "CH_TILE3D", "0123", 1),
                                                     (3, 8, "CH_TILE3D", "1", 1)])
def test_pins(ch, ctx, monkeypatch, dims, N, env, values, depth):
    rho = 0.05 + 0.02 * (np.random.default_rng(3).random(N ** dims) - 0.5)

    def run():
        s = ch.System(ctx, ch.make_desc(dims=dims, N=N, **W))
        s.upload(rho)
        s.evolve(37)
        out = s.steps_per_launch, s.region_shape, s.download()
        s.close()
        return out

    monkeypatch.delenv(env, raising=False)
    many, shape, ref = run()
    assert many > 8 and shape == (4 if dims == 2 else -1)
    for v in values:
        monkeypatch.setenv(env, v)
        k, shape, got = run()
        assert k == depth and shape == (int(v) if dims == 2 else -1)
        assert np.array_equal(got, ref)
