"""The temperature search and the resampling shared by several workgroups, at the sizes where the split
begins and where chunks and register shares end, against FP64 and the integer oracle."""
import math

import numpy as np
import pytest
import torch

from oracle import pf as opf
from oracle import rng as orng

pytestmark = pytest.mark.gpu


def _lse(v):
    m = v.max()
    return m + np.log(np.exp(v - m).sum())


def _temper(lw, lik, beta, retain, alpha, polls, schedule=None):
    from mocat_amd import _lib, transport  # noqa: F401  (registers the signatures)
    n = lw.shape[0]
    nb = _lib.c_i64(0)
    _lib.call("mocat_smc_temper_workspace_bytes", _lib.ctypes.byref(nb))
    ws = torch.full((nb.value,), 0xFF, dtype=torch.uint8, device="cuda")
    lw_d, lik_d, al = (torch.tensor(np.ascontiguousarray(v, np.float32), device="cuda") for v in (lw, lik, alpha))
    new, out = torch.empty_like(lw_d), torch.empty(8, dtype=torch.float64, device="cuda")
    _lib.call("mocat_smc_temper_split", _lib.ptr(lw_d), _lib.ptr(lik_d), n, beta, float(n), retain, 1.0, 1e-5, 1000,
              int(schedule is None), schedule or 0.0, _lib.ptr(al), alpha.shape[0], math.log(0.1), 1.0, 0.651,
              _lib.ptr(new), _lib.ptr(out), _lib.ptr(ws), nb.value, polls, _lib.stream_handle())
    return new.cpu().numpy(), out.cpu().numpy()


# around the split, a last workgroup of one particle, more workgroups' worth than the limit, more than the registers hold
@pytest.mark.parametrize("n", [1, 513, 4095, 4096, 4097, 12289, 32 * 1024 + 1, 4 * 32 * 1024 + 777])
@pytest.mark.parametrize("polls", [1 << 22, 0])  # 0: every workgroup gives up at its first wait
@pytest.mark.parametrize("retain,schedule", [(0.5, None), (0.2, None), (0.5, 0.3)])
def test_temper_split(n, polls, retain, schedule):
    rng = np.random.default_rng(n)
    lw = rng.normal(size=n).astype(np.float32)
    lik = (10 * rng.gamma(2.0, size=n)).astype(np.float32)
    if n > 5000:
        lw[4500] = -np.inf
    alpha = rng.uniform(size=(3, n)).astype(np.float32)
    new, out = _temper(lw, lik, 0.1, retain, alpha, polls, schedule)
    b = out[0]
    f0, f1 = (2 * _lse(u) - _lse(2 * u) - math.log(retain * n)
              for u in (lw.astype(np.float64) - db * lik.astype(np.float64) for db in (0.0, 0.9)))
    v = lw.astype(np.float64) - (b - 0.1) * lik.astype(np.float64)
    l1, l2 = _lse(v), _lse(2 * v)
    if schedule is not None:
        assert b == schedule
    elif f0 * f1 > 0:  # no root (the weights of lw alone retain exp(-1) of n): the nearer end
        assert b == (1.0 if abs(f1) < abs(f0) else 0.1)
    else:  # the search's stopping rule, on the log scale
        assert 0.1 < b < 1.0 and abs((2 * l1 - l2) - math.log(retain * n)) < 1e-5 + 1e-10
    # FP64 sums of at most 2^18 positive terms: relative error below 1e-11 in any order
    np.testing.assert_allclose(out[1], math.exp(2 * l1 - l2), rtol=1e-9)
    np.testing.assert_allclose(out[2:4], [l1, _lse(lw.astype(np.float64))], rtol=1e-9, atol=1e-9)
    w = np.exp(v - l1)
    am = (w * alpha.astype(np.float64).mean(0)).sum() / w.sum()
    np.testing.assert_allclose(out[4:6], [math.log(0.1) + am - 0.651, am], rtol=1e-9)
    np.testing.assert_allclose(new, v, rtol=1e-6, atol=0)


@pytest.mark.parametrize("bad,want", [(np.nan, "nan"), (np.inf, "nan"), (-np.inf, "-inf")])
def test_temper_split_non_finite(bad, want):
    n = 16384
    lw = np.full(n, bad if want == "-inf" else 0.0, np.float32)
    lw[5000] = bad
    new, out = _temper(lw, np.zeros(n, np.float32), 0.1, 0.5, np.ones((1, n), np.float32), 1 << 22, 0.3)
    assert np.isnan(out[2]) if want == "nan" else out[2] == -np.inf
    np.testing.assert_array_equal(new, lw)


@pytest.mark.parametrize("n", [4, 700, 16384])
@pytest.mark.parametrize("scale", [1.0, 3000.0])  # the larger one underflows against the chord inside the bracket
def test_temper_wide_bracket(n, scale):
    rng = np.random.default_rng(n)
    lik = (scale * rng.gamma(2.0, size=n)).astype(np.float32)
    lik[0] = 0.0
    new, out = _temper(np.zeros(n, np.float32), lik, 0.0, 0.6, np.ones((1, n), np.float32), 1 << 22)
    b = out[0]
    v = -b * lik.astype(np.float64)
    f = 2 * _lse(v) - _lse(2 * v) - math.log(0.6 * n)
    end = -lik.astype(np.float64)
    if 2 * _lse(end) - _lse(2 * end) > math.log(0.6 * n):  # no root: the ESS at 1 is still above the target
        f0 = math.log(1 / 0.6)
        assert b == (1.0 if abs(f) < f0 else 0.0)
    else:
        assert 0.0 < b < 1.0 and abs(f) < 1e-5 + 1e-10
    np.testing.assert_allclose(out[1], math.exp(2 * _lse(v) - _lse(2 * v)), rtol=1e-9)
    np.testing.assert_allclose(out[5], 1.0, rtol=1e-12)


@pytest.mark.parametrize("n", [4096, 4097, 8192, 8193, 3 * 4096 + 1, 65 * 4096 + 5])
@pytest.mark.parametrize("method", ["systematic", "multinomial"])
@pytest.mark.parametrize("kind", ["gamma", "log", "zero", "one"])
def test_resample_split(n, method, kind):
    import mocat_amd as m
    rng = np.random.default_rng(n)
    w = rng.gamma(0.3, size=n).astype(np.float32)
    if kind == "log":  # log-weights whose exponentials are exact: 0 and -inf, whole chunks of zeros among them
        w = (rng.uniform(size=n) < 0.3).astype(np.float32)
        w[4096:8192] = 0.0
        w[0] = 1.0
    elif kind == "zero":
        w[:] = 0.0
    elif kind == "one":
        w[:] = 0.0
        w[n - 1] = 3.0
    given = w
    if kind == "log":
        with np.errstate(divide="ignore"):
            given = np.log(w)
    got = m.ssm.resample_indices(torch.tensor(given, device="cuda"), m.random.PRNGKey(n), method,
                                 log_weights=kind == "log").cpu().numpy()
    if kind == "zero":
        np.testing.assert_array_equal(got, np.full(n, n - 1))  # no sum exceeds any target
    else:
        np.testing.assert_array_equal(got, opf.resample_indices(w, orng.PRNGKey(n), method))


@pytest.mark.parametrize("n", [1, 257, 4097])
@pytest.mark.parametrize("method", [-1, 0, 1, 2])
@pytest.mark.parametrize("d", [1, 20])
def test_smc_resample_keys_and_rows(n, method, d):
    """The keys of a temperature and the resampled rows, against the random and resampling entries."""
    import mocat_amd as m
    from mocat_amd import _lib, transport  # noqa: F401
    from mocat_amd.ssm.filtering import categorical
    g = torch.Generator(device="cuda").manual_seed(n)
    key = m.random.PRNGKey(n + 7)
    lw = torch.randn(n, device="cuda", generator=g)
    value, momenta = (torch.randn((n, d), device="cuda", generator=g) for _ in range(2))
    v, p, z = torch.empty_like(value), torch.empty_like(value), torch.ones_like(lw)
    mk, nk = torch.empty((n, 2), dtype=key.dtype, device="cuda"), torch.empty(2, dtype=key.dtype, device="cuda")
    nb = _lib.c_i64(0)
    _lib.call("mocat_smc_resample_workspace_bytes", n, _lib.ctypes.byref(nb))
    ws = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    _lib.call("mocat_smc_resample", _lib.ptr(key), n, d, method, *[_lib.ptr(t) for t in (lw, value, momenta, v, p, z, mk, nk)],
              _lib.ptr(ws), nb.value, _lib.stream_handle())
    keys = m.random.split(key, n + 2)
    as_int = lambda t: t.view(torch.int32)
    assert torch.equal(as_int(nk), as_int(keys[-1]))
    assert torch.equal(as_int(mk), as_int(m.random.split(keys[:n].contiguous(), 3)[:, 0].contiguous()))
    if method >= 0:
        rk = keys[n].contiguous()
        idx = categorical(rk, lw, n) if method == 2 else \
            m.ssm.resample_indices(lw, rk, ["systematic", "multinomial"][method], log_weights=True)
        assert torch.equal(v, value[idx.long()]) and torch.equal(p, momenta[idx.long()]) and not z.any()
    else:
        assert bool((z == 1).all())


@pytest.mark.parametrize("steps", [0, 1, 3])
@pytest.mark.parametrize("n,d", [(1, 1), (63, 5), (12289, 20)])
def test_smc_move_is_the_steps_it_joins(n, d, steps):
    """The joined call against evaluation, moves and temperature step called one by one: the same bits."""
    import mocat_amd as m
    from mocat_amd import _lib
    from mocat_amd.core import cdict
    rng = np.random.default_rng(n)
    sc = m.DiagonalGaussian(rng.normal(size=d), 0.5 + rng.uniform(size=d), prior_variance=4.0)
    s = m.RMMetropolisedSMCSampler(m.Underdamped(stepsize=0.3, leapfrog_steps=2, friction=0.5), mcmc_steps=steps,
                                   ess_threshold_retain=0.5)
    for k, v in s.mcmc_sampler.parameters.__dict__.items():
        if getattr(s.parameters, k, None) is None:
            setattr(s.parameters, k, v)
    beta, h = 0.123456789, 0.3
    x = torch.tensor(rng.normal(size=(n, d)), dtype=torch.float32, device="cuda")
    if n > 60:
        x[7] = math.nan
    mom = torch.tensor(rng.normal(size=(n, d)), dtype=torch.float32, device="cuda")
    keys = m.random.split(m.random.PRNGKey(3), n).contiguous()
    pp, lp, gp, gl = sc.evaluate(x, beta)
    lw = torch.tensor(rng.normal(size=n), dtype=torch.float32, device="cuda")
    one = dict(value=x.clone(), momenta=mom.clone(), grad=gp + beta * gl, pot=pp + beta * lp, pp=pp.clone(), lp=lp.clone(),
               step=torch.full((n,), h, device="cuda"), alpha=torch.ones(n, device="cuda"), keys=keys.clone(),
               trace=torch.zeros((steps, n), device="cuda"))
    X, y, packed, rows, dd, prec, pprec = sc.kernel_args()
    P = _lib.ptr
    _lib.call("mocat_hmc_lr_iterate", X, y, packed, rows, dd, prec, pprec, beta, n, P(one["value"]), P(one["momenta"]),
              P(one["grad"]), P(one["pot"]), P(one["pp"]), P(one["lp"]), P(one["step"]), P(one["alpha"]), P(one["keys"]), 0,
              steps, 2, 0.5, 1, 0.0, 1.0, 2 / 3, math.inf, None, None, P(one["trace"]), None, None, _lib.stream_handle())
    want_lw, want = s._temper(lw, one["lp"], beta, float(n), 1, math.log(h), one["trace"])
    st = cdict(value=x.clone(), momenta=mom.clone(), grad_potential=torch.empty_like(x), potential=torch.empty_like(pp),
               prior_potential=pp.clone(), likelihood_potential=lp.clone(), alpha=torch.ones(n, device="cuda"))
    trace, step, k2 = torch.zeros((steps, n), device="cuda"), torch.empty(n, device="cuda"), keys.clone()
    ws = torch.full((s._temper_args(beta, float(n), 1)[1],), 0xFF, dtype=torch.uint8, device="cuda")
    got_lw, out = s._fused_moves(sc, st, h, k2, beta, steps, trace, (gp, gl), step, lw, float(n), 1, ws)
    out = out.cpu().numpy()
    np.testing.assert_array_equal(out[:8], want)
    assert out.view(np.int64)[8] == int(torch.isnan(one["value"]).sum())
    end = one["pp"] + float(want[0]) * one["lp"]
    for a, b in [(st.value, one["value"]), (st.momenta, one["momenta"]), (st.grad_potential, one["grad"]),
                 (st.potential, end), (st.likelihood_potential, one["lp"]), (trace, one["trace"]), (got_lw, want_lw)]:
        np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
