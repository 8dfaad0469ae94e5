"""ch_set_mobility's free-energy rule M rho X^valence for the valences a system's descriptor
may not have but this call takes: zero and negative, against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,eps", [("fp64", 2.3e-16), ("fp32", 1.2e-7)])
@pytest.mark.parametrize("valence", [0, -1, -2, -5, 3])
def test_zero_and_negative_valence(ch, valence, precision, eps):
    import torch
    ctx = ch.Context(0)
    delta = 1e4 if valence >= 0 else -1e4  # 2 valence delta > 0: 0 < X <= 1
    dt = torch.float64 if precision == "fp64" else torch.float32
    rho = np.concatenate([[0.0, -0.3], np.geomspace(1e-3, 10.0, 254)])
    r = torch.tensor(rho, dtype=dt, device="cuda")
    out = torch.empty_like(r)
    torch.cuda.synchronize()
    ch.set_mobility(ctx, ch.make_desc(dims=1, N=64, precision=precision, free_energy="simple_wertheim", B2=1.0, delta=delta,
                                      valence=valence, mobility="free_energy", M=2.0), r.data_ptr(), out.data_ptr(), 256)
    ctx.synchronize()
    got, rr = out.cpu().numpy().astype(np.float64), r.cpu().numpy().astype(np.float64)
    ctx.close()
    with np.errstate(all="ignore"):
        ref = O.mobility(O.Params(dims=1, N=64, mobility=O.MOB_FREE_ENERGY, M=2.0),
                         O.Model(O.SIMPLE_WERTHEIM, B2=1.0, delta=delta, valence=valence), rr)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    n = ~np.isnan(ref)
    # a few roundings per factor of X, itself off by 1 / (c rho) <= 1 rounding and four more
    assert np.all(np.abs(got[n] - ref[n]) <= eps * (8 + 8 * abs(valence)) * np.abs(ref[n]))
