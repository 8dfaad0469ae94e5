"""f'(rho) and the free-energy mobility of SimpleWertheim outside ordinary
densities: zero, negative, denormal, infinite, NaN and below the regularisation,
against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

EDGES = np.array([0.0, -0.0, 5e-324, 1e-310, 1e-300, -1e-300, -1e-7, -1e-5, -0.3, 1e-9, 0.004999, 0.005, 0.0051, 0.7, 1e3,
                  1e30, np.inf, -np.inf, np.nan])


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


def check(got, ref, rho, valence):
    """The same special values; finite ones within 32 roundings, and the oracle's own
    error: (sqrt(1 + 2 c rho) - 1) / (c rho) loses 1 / (c rho) of its digits."""
    assert np.array_equal(np.isnan(got), np.isnan(ref)), (got, ref)
    ok = ~np.isnan(ref)
    assert np.array_equal(np.isinf(got[ok]), np.isinf(ref[ok]))
    fin = ok & np.isfinite(ref)
    assert np.all(np.sign(got[ok & ~fin]) == np.sign(ref[ok & ~fin]))
    lost = valence / np.minimum(1.0, 2.0 * valence * 1e4 * np.abs(rho[fin]))
    assert np.all(np.abs(got[fin] - ref[fin]) <= 2.3e-16 * (32 + 4 * lost) * np.maximum(1.0, np.abs(ref[fin])))


@pytest.mark.parametrize("valence", [1, 2, 4, 7])
@pytest.mark.parametrize("reg", [0.0, 0.005])
def test_edges(ch, ctx, valence, reg):
    import torch
    r = torch.tensor(np.resize(EDGES, 64), dtype=torch.float64, device="cuda")
    out = torch.empty_like(r)
    om = O.Model(O.SIMPLE_WERTHEIM, B2=1.0, delta=1e4, valence=valence, regularisation_delta=reg)
    mk = dict(free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=valence, regularisation_delta=reg)
    rho = r.cpu().numpy()
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        ch.der_bulk_free_energy(ctx, ch.make_desc(dims=1, N=64, **mk), r.data_ptr(), out.data_ptr(), r.numel())
        ctx.synchronize()
        usual = (rho > 1e-12) & (rho < 1e18) | (rho < 0) & (rho > -1e200)
        fp = out.cpu().numpy()
        check(fp[usual], O.der_bulk(om, rho)[usual], rho[usual], valence)
        print("f'", fp[:19], O.der_bulk(om, rho)[:19])
        ch.set_mobility(ctx, ch.make_desc(dims=1, N=64, mobility="free_energy", M=2.0, **mk), r.data_ptr(),
                        out.data_ptr(), r.numel())
        ctx.synchronize()
        ref = O.mobility(O.Params(dims=1, N=64, mobility=O.MOB_FREE_ENERGY, M=2.0), om, rho)
        print("mob", out.cpu().numpy()[:19], ref[:19])
        check(out.cpu().numpy()[usual], ref[usual], rho[usual], valence)
