"""Structure factor, its loss and gradient of 2D pseudospectral systems at the sizes
where the integrator keeps its spectral state line-major (N = 256 to 2048) and at
their neighbours, against the oracle; and the steps after such a call."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# one rounding of a transform of N^2 points grows with log2 N passes: 1e-10 and
# 2e-4 of the largest shell are some 1e5 and 1e2 of them, and any misplaced entry is
# of the order of the shell itself
TOL = {"fp64": 1e-10, "fp32": 2e-4}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N", [16, 128, 256, 512, 1024, 2048])
def test_structure_factor_loss_and_gradient(ch, ctx, N, precision):
    tol = TOL[precision]
    psi = O.init_density(2, N, 0.0, 0.3, 0, 11)
    target = O.radial_sq(O.init_density(2, N, 0.0, 0.3, 0, 12).reshape(N, N))
    s = ch.System(ctx, ch.make_desc(dims=2, N=N, integrator="pseudospectral", precision=precision, dt=0.01))
    s.upload(psi)
    sq = s.structure_factor()
    loss, g = s.sq_loss(target)
    s.close()
    ref = O.radial_sq(psi.reshape(N, N))
    ref_loss, ref_g = O.sq_loss(psi.reshape(N, N), target)
    assert np.abs(sq - ref).max() <= tol * ref.max()
    assert loss == pytest.approx(ref_loss, rel=10 * tol)
    assert np.abs(g - ref_g.ravel()).max() <= 10 * tol * np.abs(ref_g).max()


@pytest.mark.parametrize("N", [256, 1024])
def test_steps_after_a_structure_factor(ch, ctx, N):
    """The spectral state is not the structure factor's scratch: the same bits as without it."""
    psi = O.init_density(2, N, 0.0, 0.3, 0, 5)
    out = []
    for sq in (False, True):
        s = ch.System(ctx, ch.make_desc(dims=2, N=N, integrator="pseudospectral", dt=0.01))
        s.upload(psi)
        for _ in range(3):
            s.evolve(4)
            if sq:
                s.structure_factor()
        out.append(s.download())
        s.close()
    assert np.array_equal(*out)
