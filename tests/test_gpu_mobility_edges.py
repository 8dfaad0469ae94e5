"""The linear and regularised mobility rules bit for bit against the IEEE quotient
M rho / rho_ref and M rho / (rho + rho_min) in the system's precision: zeros, subnormals,
the ends of the range, infinities and NaN among the densities, ordinary and extreme
parameters."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(ch):
    c = ch.Context(0)
    yield c
    c.close()


def densities(dt):
    """Specials, every binade of the type, and ordinary densities."""
    fi = np.finfo(dt)
    e = np.arange(fi.minexp - fi.nmant, fi.maxexp)
    rng = np.random.default_rng(7)
    binades = np.ldexp((1 + rng.random((8, e.size))).astype(dt), e).ravel()
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, fi.max, -fi.max, fi.tiny, -fi.tiny, fi.smallest_subnormal,
                        -fi.smallest_subnormal], dtype=dt)
    return np.concatenate([special, binades, -binades, rng.random(4096).astype(dt)]).astype(dt)


def same(got, ref):
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    i = np.uint64 if got.dtype == np.float64 else np.uint32
    n = ~np.isnan(ref)
    bad = got[n].view(i) != ref[n].view(i)
    assert not bad.any(), (got[n][bad][:8], ref[n][bad][:8])


@pytest.mark.parametrize("par", [0.05, 1.0, 3.0, -0.7, 1e-30, 1e30, 1e-39, 1e-310, 1e300, np.inf, 0.0])
@pytest.mark.parametrize("rule", ["linear", "regularised"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_quotient_rules(ch, ctx, precision, rule, par):
    import torch
    dt = np.float64 if precision == "fp64" else np.float32
    rho = densities(dt)
    r = torch.from_numpy(rho).cuda()
    out = torch.empty_like(r)
    torch.cuda.synchronize()
    M = dt(1.7)
    key = "rho_ref" if rule == "linear" else "rho_min"
    ch.set_mobility(ctx, ch.make_desc(dims=1, N=64, precision=precision, mobility=rule, M=float(M), **{key: par}),
                    r.data_ptr(), out.data_ptr(), r.numel())
    ctx.synchronize()
    with np.errstate(all="ignore"):
        ref = M * rho / (dt(par) if rule == "linear" else rho + dt(par))
    assert ref.dtype == dt
    same(out.cpu().numpy(), ref)


@pytest.mark.parametrize("dims,N", [(1, 64), (2, 16), (2, 64), (2, 128), (3, 8), (3, 32)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("rho_ref", [1.5, -1.5])
@pytest.mark.parametrize("end", ["tiny", "huge"])
def test_steps_with_an_extreme_reference_density(ch, ctx, dims, N, precision, rho_ref, end):
    """M and rho_ref scaled by one power of two give the same bits, also where rho_ref
    is subnormal or its reciprocal is."""
    e = {("fp64", "tiny"): -1023, ("fp64", "huge"): 1023, ("fp32", "tiny"): -128, ("fp32", "huge"): 127}[precision, end]
    rho = 0.05 + 0.02 * (np.random.default_rng(3).random(N ** dims) - 0.5)
    out = []
    for s in (0, e):
        # M far enough from the ends of the range: the numerators stay normal
        M, ref = (2.0 ** 10, rho_ref) if end == "tiny" else (2.0 ** -10, rho_ref)
        sy = ch.System(ctx, ch.make_desc(dims=dims, N=N, integrator="euler_mobility", mobility="linear", dt=1e-4,
                                         precision=precision, M=float(np.ldexp(M, s)), rho_ref=float(np.ldexp(ref, s))))
        sy.upload(rho)
        sy.evolve(3)
        out.append(sy.download())
        sy.close()
    assert np.isfinite(out[0]).all()
    assert np.array_equal(*out)
