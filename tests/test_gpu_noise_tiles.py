"""Every tile of the conserved-noise step (CH_NOISE_TILE) and the default, which depends on
dims, N, precision and mobility, give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RULES = {"constant": {}, "regularised": dict(rho_min=0.5), "linear": dict(rho_ref=0.5)}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("dims,N", [(2, 64), (2, 512), (2, 1024), (3, 16), (3, 32), (3, 64), (3, 128)])
def test_tiles_agree(ch, ctx, monkeypatch, dims, N, rule, precision):
    rho = 0.3 + 0.1 * (np.random.default_rng(N).random(N ** dims) - 0.5)
    out = []
    for tile in (None, "0", "1", "2"):
        if tile is None:
            monkeypatch.delenv("CH_NOISE_TILE", raising=False)
        else:
            monkeypatch.setenv("CH_NOISE_TILE", tile)
        s = ch.System(ctx, ch.make_desc(dims=dims, N=N, precision=precision, integrator="euler_mobility", mobility=rule,
                                        dt=1e-3, with_noise=True, noise_rescale_factor=1e-2, seed=9, **RULES[rule]))
        s.upload(rho)
        s.evolve(3)
        out.append(s.download())
        s.close()
    assert np.isfinite(out[0]).all() and not np.array_equal(out[0], rho)
    for o in out[1:]:
        assert np.array_equal(o, out[0])
