"""Generic multi-species models of every size class against the oracle: 1 to 4
patch types with all of them carried (register-resident vectors), a patch type
that no species carries and a fifth species (run-time indexed vectors).

Tolerance 1e-8 relative: a cell's mass-action sweeps stop once none of its X
moves by 1e-8, and round-off can move the stop by one sweep.  A step count that
recurs replays a captured chain: the same bits as direct steps."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_linf

pytestmark = pytest.mark.gpu

MODELS = {
    "P1": ([[0] * 4], {(0, 0): 900.0}),
    "P2": ([[0] * 5, [1] * 2, [0, 1, 1]], {(0, 0): 1e3, (0, 1): 200.0, (1, 1): 2e3}),
    "P3": ([[0, 1], [1, 2, 2]], {(0, 1): 700.0, (1, 2): 300.0, (2, 2): 150.0}),
    "P4_S4": ([[0, 0], [1], [2, 2, 3], [3, 3, 3]], {(0, 1): 800.0, (2, 3): 500.0, (0, 0): 100.0, (3, 3): 60.0}),
    "gap": ([[0, 0], [2, 2, 0]], {(0, 0): 400.0, (0, 2): 300.0, (1, 2): 999.0}),
    "S5": ([[0, 0], [1], [0, 1], [1, 1], [0]], {(0, 1): 800.0, (0, 0): 100.0}),
}


def build(name, cls):
    patches, deltas = MODELS[name]
    S = len(patches)
    return O.generic_model(tuple(1.0 + 0.2 * i for i in range(S)), patches, deltas,
                           {(a, b): 0.3 + 0.1 * (a + b) for a in range(S) for b in range(a, S)}, model_cls=cls)


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("name", list(MODELS))
@pytest.mark.parametrize("N", [8, 32])
def test_generic_sizes(ch, ctx, name, N):
    om, gm = build(name, O.SpeciesModel), build(name, ch.ChSpeciesModel)
    p = O.Params(dims=2, N=N, dt=1e-4, dx=1.0, k=1.0, mobility=O.MOB_FREE_ENERGY, M=1.0)
    desc = ch.make_desc(dims=2, N=N, integrator="euler_mobility", free_energy="generic_wertheim", dt=1e-4, dx=1.0,
                        M=1.0, mobility="free_energy")
    rng = np.random.default_rng(5)
    rho0 = 0.03 * (1 + 0.2 * (2 * rng.random(om.n_species * N * N) - 1))
    want = O.run_ms(O.EULER_MOBILITY, p, om, rho0, 21)
    got = []
    for splits in ((21,), (7, 7, 7)):
        s = ch.System(ctx, desc, species_model=gm)
        s.upload(rho0)
        for n in splits:
            s.evolve(n)
        got.append(s.download())
        s.close()
    err = rel_linf(got[0], want)
    print(f"{name} N={N}: rel L-inf vs oracle = {err:.3e}")
    assert err < 1e-8
    assert np.array_equal(got[0], got[1])
