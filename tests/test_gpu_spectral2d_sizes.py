"""The 2D pseudospectral chain at every grid size up to 512 (each column engine and
row packing: several lines or rows per block, one, two waves per line) against the
oracle, over calls that begin and end a chain."""
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


@pytest.mark.parametrize("N", [4, 8, 16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("dealias", [False, True])
def test_chain_against_oracle(ch, ctx, N, dealias):
    """FP64 within 1e-12 relative L-inf of the oracle (12 steps, each two transforms
    of some log2(N^2) <= 18 roundings of 1.1e-16: below 1e-13, taken ten times); FP32
    within 12 * 2 * 18 * 6e-8 = 2.6e-5."""
    rho0 = O.init_density(2, N, 0.1, 0.3, 0, 31 + N)
    kw = dict(dims=2, N=N, dt=0.05, dx=1.0, k=1.0, M=1.0, S=0.4)
    ref = O.run(O.PSEUDOSPECTRAL, O.Params(use_dealias=int(dealias), **kw), O.Model(epsilon=0.9), rho0, 12)
    for precision, tol in (("fp64", 1e-12), ("fp32", 2.6e-5)):
        s = ch.System(ctx, ch.make_desc(integrator="pseudospectral", precision=precision, epsilon=0.9,
                                        use_dealias=dealias, **kw))
        s.upload(rho0)
        for n in (1, 4, 7):
            s.evolve(n)
        err = rel_linf(s.download(), ref)
        s.close()
        print(f"N={N} {precision} rel L-inf {err:.2e}", flush=True)
        assert err < tol
