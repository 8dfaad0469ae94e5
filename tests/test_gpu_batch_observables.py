"""Observables of batches on both sides of the rule for one block per replica (Landau
replicas of N = 64 alone, 1024 replicas and more) or several, against single systems."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MODELS = {"landau": dict(dt=0.01), "wertheim": dict(free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=4, dt=1e-4)}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("model", list(MODELS))
@pytest.mark.parametrize("sizes", [[64], [64] * 3, [64, 128], [512, 64], [64] * 1023, [64] * 1024],
                         ids=["1x64", "3x64", "64_128", "512_64", "1023x64", "1024x64"])
def test_batch_observables(ch, ctx, sizes, model, precision):
    kw = dict(dims=2, precision=precision, **MODELS[model])
    b = ch.Batch(ctx, [ch.make_desc(N=N, **kw) for N in sizes])
    fields = [0.05 + 0.02 * (np.random.default_rng(r % 7).random(N * N) - 0.5) for r, N in enumerate(sizes)]
    for r, f in enumerate(fields):
        b.upload(r, f)
    mass, fe = b.observables()
    b.close()
    ref = {}
    for r, N in enumerate(sizes):
        key = (r % 7, N)
        if key not in ref:
            s = ch.System(ctx, ch.make_desc(N=N, **kw))
            s.upload(fields[r])
            ref[key] = s.observables()
            s.close()
        # FP64 sums of at most 2^18 cells of one sign, in two orders
        assert mass[r] == pytest.approx(ref[key][0], rel=1e-13)
        assert fe[r] == pytest.approx(ref[key][1], rel=1e-12)
