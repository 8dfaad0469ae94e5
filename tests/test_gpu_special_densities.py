"""f' and the free-energy mobility of SimpleWertheim at zero, subnormal, tiny, huge,
infinite and NaN densities: the oracle's special values, and for tiny positive densities,
where its (sqrt(1 + 2 c rho) - 1) / (c rho) cancels to 0, the limit X = 1."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

TINY = np.array([5e-324, 1e-310, 2.3e-308, 1e-300, 1e-200])
OTHER = np.array([0.0, -0.0, 1e19, 1e30, 1e100, np.inf, -np.inf, np.nan])
DELTA = 1e4


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


def pointwise(ctx, call, desc, rho):
    import torch
    r = torch.tensor(rho, dtype=torch.float64, device="cuda")
    out = torch.empty_like(r)
    torch.cuda.synchronize()
    call(ctx, desc, r.data_ptr(), out.data_ptr(), r.numel())
    ctx.synchronize()
    return out.cpu().numpy()


def same_or_close(got, ref, roundings):
    assert np.array_equal(np.isnan(got), np.isnan(ref)), (got, ref)
    inf = np.isinf(ref)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], ref[inf]), (got, ref)
    fin = np.isfinite(ref)
    assert np.all(np.abs(got[fin] - ref[fin]) <= 2.3e-16 * roundings * np.abs(ref[fin])), (got, ref)


@pytest.mark.parametrize("valence", [1, 2, 4, 7])
@pytest.mark.parametrize("reg", [0.0, 0.005])
def test_fprime(ch, ctx, valence, reg):
    desc = ch.make_desc(dims=1, N=64, free_energy="simple_wertheim", B2=1.0, delta=DELTA, valence=valence,
                        regularisation_delta=reg)
    om = O.Model(O.SIMPLE_WERTHEIM, B2=1.0, delta=DELTA, valence=valence, regularisation_delta=reg)
    with np.errstate(all="ignore"):
        # three terms, a logarithm within 2 ulp and products of `valence` factors
        same_or_close(pointwise(ctx, ch.der_bulk_free_energy, desc, OTHER), O.der_bulk(om, OTHER), 16 + 4 * valence)
        # X = 1 - c rho + ..., below 1e-190 from 1: ln X vanishes
        limit = np.log(TINY) if reg == 0.0 else np.log(reg) + (TINY - reg) / reg
        same_or_close(pointwise(ctx, ch.der_bulk_free_energy, desc, TINY), limit + 2.0 * TINY, 16)


@pytest.mark.parametrize("valence", [1, 2, 4, 7])
def test_free_energy_mobility(ch, ctx, valence):
    M = 2.0
    desc = ch.make_desc(dims=1, N=64, free_energy="simple_wertheim", B2=1.0, delta=DELTA, valence=valence,
                        mobility="free_energy", M=M)
    om = O.Model(O.SIMPLE_WERTHEIM, B2=1.0, delta=DELTA, valence=valence)
    op = O.Params(dims=1, N=64, mobility=O.MOB_FREE_ENERGY, M=M)
    with np.errstate(all="ignore"):
        same_or_close(pointwise(ctx, ch.set_mobility, desc, OTHER), O.mobility(op, om, OTHER), 16 + 8 * valence)
    same_or_close(pointwise(ctx, ch.set_mobility, desc, TINY), M * TINY, 4)
