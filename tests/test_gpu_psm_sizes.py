"""The fused splitting chain of pseudospectral_mobility at the sizes where its
line engines and row packing change (2D N = 4 .. 512, 4096; 3D N = 4 .. 32),
against the element-wise kernels around whole transforms (CH_PSM_FUSE=0): the
same operations, with transforms of another factorisation at some sizes, so
round-off apart: <= 1e-12 relative after 7 steps (FP64; each transform's error
is a few 1e-16), 1e-5 in FP32."""
import numpy as np
import pytest

from helpers import rel_linf

pytestmark = pytest.mark.gpu

SIZES = [(2, 4), (2, 8), (2, 32), (2, 128), (2, 256), (2, 512), (2, 4096), (3, 4), (3, 8), (3, 32)]
RULES = {"regularised": ("landau", dict(rho_min=0.2), 0.5), "linear": ("simple_wertheim", dict(rho_ref=0.05), 0.05),
         "free_energy": ("simple_wertheim", {}, 0.05)}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("rule", list(RULES))
@pytest.mark.parametrize("dims,N", SIZES, ids=[f"{d}d_N{n}" for d, n in SIZES])
def test_fused_chain_sizes(ch, ctx, monkeypatch, dims, N, rule, precision):
    if N == 4096 and (rule != "regularised" or precision == "fp32"):
        pytest.skip("one combination at the largest grid")
    print(f"case {dims}D N={N} {rule} {precision}", flush=True)
    model, kw, base = RULES[rule]
    rng = np.random.default_rng(N + dims)
    rho0 = base * (1 + 0.1 * (2 * rng.random(N ** dims) - 1))
    desc = ch.make_desc(dims=dims, N=N, integrator="pseudospectral_mobility", free_energy=model, mobility=rule,
                        precision=precision, dt=0.01 if model == "landau" else 1e-4, dx=0.9, k=1.0, S=0.3, delta=1e4,
                        use_dealias=dims == 2, **kw)
    out = {}
    for fuse, splits in (("1", (3, 3, 1)), ("0", (7,))):
        monkeypatch.setenv("CH_PSM_FUSE", fuse)
        s = ch.System(ctx, desc)
        s.upload(rho0)
        for n in splits:
            s.evolve(n)
        out[fuse] = s.download()
        s.close()
    err = rel_linf(out["1"], out["0"])
    print(f"rel L-inf fused vs element-wise = {err:.3e}")
    assert err < (1e-12 if precision == "fp64" else 1e-5)
