"""The 3D euler_mobility reverse step in one launch marching along z (CH_TILE3D=5)
against the two-launch form (3), at the sizes of its three block shapes; and a
record whose last window stays on its tape against one swept a second time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = dict(integrator="euler_mobility", free_energy="simple_wertheim", B2=1.0, delta=1e4, valence=4, dt=1e-4, k=1.0)
CASES = {
    "constant": dict(**W),
    "linear": dict(mobility="linear", rho_ref=0.05, **W),
    "regularised": dict(mobility="regularised", rho_min=0.1, **W),
}


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("N,ckpt", [(32, 0), (32, 2), (64, 0), (64, 3), (128, 0)])
def test_march_reverse_equals_two_launches(ch, ctx, monkeypatch, N, ckpt, case, precision):
    """lambda and psi bit for bit; the gradients sum 5 N^3 FP64 terms in another
    order: within n^1/2 ulp of the sum of magnitudes, taken 1e-9 of the largest."""
    from cahn_hilliard_amd.init import initial_density
    print(f"case {case} N={N} ckpt={ckpt} {precision}", flush=True)
    got = []
    for t3 in ("5", "3"):
        monkeypatch.setenv("CH_TILE3D", t3)
        s = ch.System(ctx, ch.make_desc(dims=3, N=N, precision=precision, **CASES[case]))
        s.upload(initial_density(3, N, 0.05, 0.05, 0, 99 + N))
        s.record(5, ckpt)
        got.append((s.download(), *s.adjoint(np.cos(np.arange(N ** 3)))))
        s.close()
    for a, b in zip(got[0][:2], got[1][:2]):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
    assert np.abs(got[0][2] - got[1][2]).max() <= 1e-9 * np.abs(got[1][2]).max()


@pytest.mark.parametrize("dims,N,kw", [(1, 256, dict(dt=0.004)), (2, 32, dict(dt=0.004)), (2, 128, dict(dt=0.004)),
                                       (2, 64, CASES["linear"]), (3, 16, CASES["regularised"]), (3, 32, CASES["linear"])])
@pytest.mark.parametrize("steps,ckpt", [(1, 1), (7, 7), (9, 5), (10, 5), (23, 5), (24, 8)])
def test_last_window_stays_on_its_tape(ch, ctx, dims, N, kw, steps, ckpt):
    """One to five windows, the last one whole or short: the end state of evolve, the
    lambda of a sweep over every kept state, and lambda and gradients again from a
    second sweep, which recomputes the windows whose buffer was taken (the gradients
    are summed launch by launch, so their bits depend on the windows)."""
    rho = 0.05 + 0.01 * np.random.default_rng(N + steps).random(N ** dims)
    w = np.cos(np.arange(N ** dims))
    s = ch.System(ctx, ch.make_desc(dims=dims, N=N, **kw))
    s.upload(rho)
    s.evolve(steps)
    end = s.download()
    s.upload(rho)
    s.record(steps, 0)
    ref = s.adjoint(w)
    s.upload(rho)
    s.record(steps, ckpt)
    assert np.array_equal(s.download(), end)
    first, second = s.adjoint(w), s.adjoint(w)
    assert np.array_equal(first[0], ref[0]) and np.array_equal(second[0], ref[0])
    assert np.array_equal(first[1], second[1])
    s.close()
