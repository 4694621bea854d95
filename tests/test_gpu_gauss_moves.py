"""One update of the diagonal Gaussian's move kernel against FP64 on the same keys, at the column counts where the lanes
per chain change and at ragged chain counts."""
import math

import numpy as np
import pytest
import torch

from oracle import rng as orng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [1, 2, 8, 9, 16, 17, 20, 32, 33, 64, 65, 100, 128])
@pytest.mark.parametrize("correction", [0, 1, 2])
@pytest.mark.parametrize("flat", [False, True])
def test_one_update(d, correction, flat):
    import mocat_amd as m
    from mocat_amd import _lib, transport  # noqa: F401  (registers the signatures)
    C, L, beta, friction, prec = 37, 3, 0.3, 0.7, 0.0 if flat else 0.1
    rs = np.random.default_rng(d)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)
    mu, lam = f32(rs.normal(size=d)), f32(1 / rs.uniform(0.3, 2.0, d))
    x, p, step = f32(rs.normal(size=(C, d))), f32(rs.normal(size=(C, d))), f32(rs.uniform(0.05, 0.2, C))
    keys = np.asarray(orng.split(orng.PRNGKey(d), C), np.uint32)
    u64 = lambda a: a.astype(np.float64)

    def potential(v):
        lik = 0.5 * (u64(lam) * (v - u64(mu)) ** 2).sum(1)
        pri = 0.5 * prec * (v ** 2).sum(1) + (0.0 if flat else 0.5 * d * (math.log(2 * math.pi) - math.log(prec)))
        return pri, lik, prec * v + beta * u64(lam) * (v - u64(mu))

    pri0, lik0, g0 = potential(u64(x))
    # the kernel's inputs, rounded once
    t = lambda a: torch.tensor(f32(a), device="cuda")
    th, mom, grad, prior, lik, pot, st = t(x), t(p), t(g0), t(pri0), t(lik0), t(pri0 + beta * lik0), t(step)
    alpha, k = torch.zeros(C, device="cuda"), torch.tensor(keys.astype(np.int64), device="cuda").to(torch.uint32)
    tr = {n: torch.zeros((1, C, d) if n in ("v", "m") else (1, C), device="cuda") for n in ("v", "u", "a", "s", "m")}
    P = _lib.ptr
    mu_d, lam_d = t(mu), t(lam)
    _lib.call("mocat_hmc_lr_iterate", P(mu_d), P(lam_d), None, 1, d, 2, prec, beta, C, P(th), P(mom), P(grad), P(pot),
              P(prior), P(lik), P(st), P(alpha), P(k), 0, 1, L, friction, correction, 0.65, 1.0, 2 / 3, math.inf,
              *[P(tr[n]) for n in ("v", "u", "a", "s", "m")], _lib.stream_handle())
    # the same update in FP64
    z, u, kend = np.empty((C, d)), np.empty(C), np.empty((C, 2), np.uint32)
    for c in range(C):
        nk, sub = orng.split(keys[c], 2)
        z[c] = orng.normal(sub, (d,))
        nk = orng.split(nk, L + 1)[0]
        if correction:
            nk, sub = orng.split(nk, 2)
            u[c] = orng.uniform(sub)
        kend[c] = nk
    h = u64(step)[:, None]
    q = -u64(p) * np.exp(-friction * h) + np.sqrt(1 - np.exp(-2 * friction * h)) * z
    v, w, g = u64(x), q, u64(f32(g0))
    for _ in range(L):
        w = w - h / 2 * g
        v = v + h * w
        pri, lk, g = potential(v)
        w = w - h / 2 * g
    kin = lambda a: 0.5 * (a ** 2).sum(1)
    a = np.minimum(1.0, np.exp(-(pri + beta * lk) + (pri0 + beta * lik0) - kin(w) + kin(q))) if correction else np.ones(C)
    acc = u < a if correction else np.ones(C, bool)
    np.testing.assert_array_equal(k.cpu().numpy().astype(np.uint32), kend)
    # potentials are sums of d terms of magnitude below 100 in f32: absolute error of the exponent below d * 1e-5
    np.testing.assert_allclose(alpha.cpu().numpy(), a, atol=1e-4 + d * 1e-5)
    sure = np.abs(u - a) > 1e-3 + d * 1e-4 if correction else np.ones(C, bool)
    assert sure.mean() > 0.8
    pick = lambda new, old: np.where((acc if new.ndim == 1 else acc[:, None]), new, old)[sure]
    close = lambda got, want: np.testing.assert_allclose(got.cpu().numpy()[sure], want, rtol=2e-5, atol=2e-5)
    close(th, pick(v, u64(x)))
    close(mom, pick(-w, q))
    close(grad, pick(g, g0))
    np.testing.assert_allclose(lik.cpu().numpy()[sure], pick(lk, lik0), rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(prior.cpu().numpy()[sure], pick(pri, pri0), rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(pot.cpu().numpy()[sure], pick(pri + beta * lk, pri0 + beta * lik0), rtol=1e-4, atol=1e-4)
    want = np.log(u64(step)) + (a - 0.65) if correction == 2 else np.log(u64(step))
    np.testing.assert_allclose(np.log(st.cpu().numpy()), want, atol=2e-4 + d * 1e-5)
    for n, full in (("v", th), ("u", pot), ("a", alpha), ("s", st), ("m", mom)):
        assert torch.equal(tr[n][0], full)
