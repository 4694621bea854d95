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
@pytest.mark.parametrize("n", [1, 12287, 12288, 12289, 32 * 1024 + 1, 4 * 32 * 1024 + 777])
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
