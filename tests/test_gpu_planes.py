"""3D pseudospectral chains whose x and y passes run as one plane per block
(N = 32, 64; 128 in FP32): against the oracle at N = 32 (<= 1e-10 relative after
12 steps, dealiasing and S on and off), and split anywhere with the same bits."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_linf

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


def start(N, base=0.0):
    rng = np.random.default_rng(N)
    return base + (0.05 if base == 0.0 else 0.2 * base) * (2 * rng.random(N ** 3) - 1)


@pytest.mark.parametrize("S,dealias", [(0.0, False), (0.4, True)])
@pytest.mark.parametrize("model", ["landau", "simple_wertheim"])
def test_planes_match_oracle(ch, ctx, model, S, dealias):
    N, dt = 32, 0.05 if model == "landau" else 1e-3
    rho0 = start(N, 0.0 if model == "landau" else 0.05)
    om = O.Model(epsilon=0.9) if model == "landau" else O.Model(O.SIMPLE_WERTHEIM, B2=1.0, delta=1e4, valence=4)
    want = O.run(O.PSEUDOSPECTRAL, O.Params(dims=3, N=N, dt=dt, dx=1.1, k=1.0, S=S, use_dealias=int(dealias)), om, rho0, 12)
    s = ch.System(ctx, ch.make_desc(dims=3, N=N, integrator="pseudospectral", free_energy=model, dt=dt, dx=1.1, S=S,
                                    use_dealias=dealias))
    s.upload(rho0)
    s.evolve(12)
    err = rel_linf(s.download(), want)
    s.close()
    print(f"{model} S={S} dealias={dealias}: rel L-inf vs oracle = {err:.3e}")
    assert err < 1e-10


@pytest.mark.parametrize("N,precision", [(32, "fp64"), (32, "fp32"), (64, "fp64"), (64, "fp32"), (128, "fp32")])
@pytest.mark.parametrize("model", ["landau", "simple_wertheim"])
def test_plane_chains_split(ch, ctx, N, precision, model):
    rho0 = start(N, 0.0 if model == "landau" else 0.05)
    out = []
    for splits in ((7,), (1, 2, 4)):
        s = ch.System(ctx, ch.make_desc(dims=3, N=N, integrator="pseudospectral", free_energy=model,
                                        precision=precision, dt=0.05 if model == "landau" else 1e-3))
        s.upload(rho0)
        for n in splits:
            s.evolve(n)
        out.append(s.download())
        s.close()
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])
