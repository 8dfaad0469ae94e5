"""FP32 and large-grid forms of the spectral passes against the FP64 oracle: 3D planes at
N = 64 and 128 in FP32, the multi-species column pass in FP32 at every engine and at N =
2048 in both precisions.

FP32 tolerance: a transform of 2^21 points is off by at most 21 roundings of 6e-8, 1.3e-6
of the field; 4 steps of two transforms each and the roundings between them stay
below 2e-5.  FP64: 1e-10, as the other tests of these steps."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_linf
from test_gpu_species import ricci, setup

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-10, "fp32": 2e-5}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("model", ["landau", "simple_wertheim"])
@pytest.mark.parametrize("N", [64, 128])
def test_planes_fp32(ch, ctx, N, model):
    base, dt = (0.3, 0.05) if model == "landau" else (0.05, 1e-3)
    rho0 = base * (1 + 0.2 * (2 * np.random.default_rng(N).random(N ** 3) - 1))
    om = O.Model(epsilon=0.9) if model == "landau" else O.Model(O.SIMPLE_WERTHEIM, B2=1.0, delta=1e4, valence=4)
    want = O.run(O.PSEUDOSPECTRAL, O.Params(dims=3, N=N, dt=dt, dx=1.1, k=1.0, S=0.4), om, rho0, 4)
    s = ch.System(ctx, ch.make_desc(dims=3, N=N, integrator="pseudospectral", free_energy=model, precision="fp32", dt=dt,
                                    dx=1.1, S=0.4))
    s.upload(rho0)
    s.evolve(1)
    s.evolve(3)
    err = rel_linf(s.download(), want)
    s.close()
    print(f"N={N} {model}: rel L-inf {err:.2e}", flush=True)
    assert err < TOL["fp32"]


@pytest.mark.parametrize("N,precision,steps", [(8, "fp32", 4), (128, "fp32", 4), (256, "fp32", 4), (512, "fp32", 4),
                                               (1024, "fp32", 4), (2048, "fp32", 2), (2048, "fp64", 2)])
def test_species_columns(ch, ctx, N, precision, steps):
    case = ("ps", ricci, "pseudospectral", 2, N, 1e-3, dict(mobility="constant"), 0.3, True)
    om, gm, p, desc, rho0 = setup(ch, case)
    desc.precision = ch.FP32 if precision == "fp32" else ch.FP64
    want = O.run_ms(O.PSEUDOSPECTRAL, p, om, rho0, steps)
    s = ch.System(ctx, desc, species_model=gm)
    s.upload(rho0)
    s.evolve(steps)
    err = rel_linf(s.download(), want)
    s.close()
    print(f"N={N} {precision}: rel L-inf {err:.2e}", flush=True)
    assert err < TOL[precision]
