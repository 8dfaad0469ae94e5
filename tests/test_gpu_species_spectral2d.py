"""The multi-species 2D pseudospectral step at every column engine's sizes (several
lines per block, one wave, two waves per line), with a k of its own for each
species, against the oracle: 1e-10 relative, as the models' other fields (analytic
X, FP64)."""
import pytest

import oracle as O
from helpers import rel_linf
from test_gpu_species import ricci, setup

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("dealias", [False, True])
@pytest.mark.parametrize("N", [4, 8, 32, 128, 256, 512, 1024])
def test_column_pass_sizes(ch, ctx, N, dealias):
    case = ("ps", ricci, "pseudospectral", 2, N, 1e-3, dict(mobility="constant"), 0.3, dealias)
    om, gm, p, desc, rho0 = setup(ch, case)
    want = O.run_ms(O.PSEUDOSPECTRAL, p, om, rho0, 5)
    s = ch.System(ctx, desc, species_model=gm)
    s.upload(rho0)
    s.evolve(2)
    s.evolve(3)
    err = rel_linf(s.download(), want)
    s.close()
    print(f"N={N} dealias={dealias}: rel L-inf {err:.2e}", flush=True)
    assert err < 1e-10
