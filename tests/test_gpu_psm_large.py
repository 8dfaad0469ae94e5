"""The splitting step of pseudospectral_mobility on large grids: 3D N = 128 and 256, whose
row packing and partial maxima differ from the small ones', 2D FP32 N = 2048 and 4096
(fused passes) and FP64 N = 2048 (whole transforms, fused divergence), against the
element-wise kernels around whole transforms (CH_PSM_FUSE=0).  The same operations with
transforms of another factorisation: <= 1e-12 relative after 5 steps in FP64 (each
transform's error is a few 1e-16), 1e-5 in FP32."""
import numpy as np
import pytest

from helpers import rel_linf

pytestmark = pytest.mark.gpu

RULES = {"regularised": ("landau", dict(rho_min=0.2), 0.5), "free_energy": ("simple_wertheim", {}, 0.05)}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("dims,N,precision", [(3, 128, "fp64"), (3, 128, "fp32"), (3, 256, "fp64"), (2, 2048, "fp64"),
                                              (2, 2048, "fp32"), (2, 4096, "fp32")])
def test_large_grids(ch, ctx, monkeypatch, dims, N, precision, rule):
    print(f"case {dims}D N={N} {rule} {precision}", flush=True)
    model, kw, base = RULES[rule]
    rho0 = base * (1 + 0.1 * (2 * np.random.default_rng(N + dims).random(N ** dims) - 1))
    desc = ch.make_desc(dims=dims, N=N, integrator="pseudospectral_mobility", free_energy=model, mobility=rule,
                        precision=precision, dt=0.01 if model == "landau" else 1e-4, dx=0.9, k=1.0, S=0.3, delta=1e4,
                        use_dealias=dims == 2, **kw)
    out = {}
    for fuse, splits in (("1", (2, 2, 1)), ("0", (5,))):
        monkeypatch.setenv("CH_PSM_FUSE", fuse)
        s = ch.System(ctx, desc)
        s.upload(rho0)
        for n in splits:
            s.evolve(n)
        out[fuse] = s.download()
        s.close()
    assert np.isfinite(out["0"]).all() and not np.array_equal(out["0"], rho0)
    assert rel_linf(out["1"], out["0"]) < (1e-12 if precision == "fp64" else 1e-5)
