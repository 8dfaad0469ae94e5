"""The 3D step marching along z (CH_TILE3D=4) against the fused LDS tile (1), bit
for bit, at the sizes of its three block shapes and with every mobility rule:
both evaluate each cell with the same arithmetic.  And the default choice
records and sweeps back with the bits of the two-launch forms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = dict(free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=4, dt=1e-4)
CASES = {
    "landau_euler": dict(integrator="euler", dt=0.004),
    "landau_em_constant": dict(integrator="euler_mobility", dt=0.004, dx=0.9),
    "landau_em_regularised": dict(integrator="euler_mobility", mobility="regularised", rho_min=0.5, dt=1e-3),
    "wertheim_euler": dict(integrator="euler", **W),
    "wertheim_em_linear": dict(integrator="euler_mobility", mobility="linear", rho_ref=0.05, **W),
    "wertheim_em_regularised": dict(integrator="euler_mobility", mobility="regularised", rho_min=0.1, **W),
    "wertheim_em_free_energy": dict(integrator="euler_mobility", mobility="free_energy", **W),
}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


def start(case, N):
    from cahn_hilliard_amd.init import initial_density
    return initial_density(3, N, 0.3 if "landau" in case else 0.05, 0.05, 0, 99 + N)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("N", [32, 64, 128])
def test_march_equals_tile(ch, ctx, monkeypatch, N, case, precision):
    print(f"case {case} N={N} {precision}", flush=True)
    out = {}
    for t3 in ("1", "4"):
        monkeypatch.setenv("CH_TILE3D", t3)
        s = ch.System(ctx, ch.make_desc(dims=3, N=N, precision=precision, k=1.0, **CASES[case]))
        s.upload(start(case, N))
        s.evolve(9)
        out[t3] = s.download()
        s.close()
    assert np.all(np.isfinite(out["4"])) and np.array_equal(out["1"], out["4"])


@pytest.mark.parametrize("case", ["landau_em_regularised", "wertheim_em_linear", "wertheim_em_free_energy"])
@pytest.mark.parametrize("ckpt", [0, 4])
def test_march_reverse_mode(ch, ctx, monkeypatch, case, ckpt):
    print(f"case {case} ckpt={ckpt}", flush=True)
    N, got = 32, []
    for t3 in (None, "1"):
        if t3:
            monkeypatch.setenv("CH_TILE3D", t3)
        s = ch.System(ctx, ch.make_desc(dims=3, N=N, k=1.0, **CASES[case]))
        s.upload(start(case, N))
        s.record(9, ckpt)
        _, seed, _ = s.free_energy_grad()
        lam, grads = s.adjoint(seed)
        got.append((s.download(), lam, grads))
        s.close()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert np.abs(got[0][2] - got[1][2]).max() <= 1e-12 * np.abs(got[1][2]).max()
