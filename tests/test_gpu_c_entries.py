"""Entries of the C interface that the package itself does not call: the kernel Stein discrepancy's row sums and the
temperature step by one workgroup."""
import math

import numpy as np
import pytest
import torch

from oracle import ksd as ok

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,shares", [(1, 1, 1), (65, 33, 2), (200, 7, 4)])
@pytest.mark.parametrize("kernel,prm", [("gaussian", {}), ("imq", dict(c=1.0, beta=-0.5)), ("imq", dict(c=1.5, beta=-0.75))])
@pytest.mark.parametrize("weighted", [False, True])
def test_ksd_rows(n, d, shares, kernel, prm, weighted):
    from mocat_amd import _lib, metrics  # noqa: F401  (registers the signature)
    rs = np.random.default_rng(n)
    x = rs.normal(0.5, 1.2, (n, d)).astype(np.float32)
    g = (0.8 * x + rs.normal(0, 0.3, (n, d))).astype(np.float32)
    w = rs.uniform(0.5, 2.0, n).astype(np.float32)
    h = float(np.float32(0.7 * math.sqrt(d)))
    xd, gd, wd = (torch.tensor(t, device="cuda") for t in (x, g, w))
    part = torch.full((shares, n), np.nan, dtype=torch.float64, device="cuda")
    _lib.call("mocat_ksd_rows", _lib.ptr(xd), _lib.ptr(gd), _lib.ptr(wd if weighted else None), n, d, int(kernel == "imq"), h,
              prm.get("c", 1.0), prm.get("beta", -0.5), shares, _lib.ptr(part), _lib.stream_handle())
    x, g = x.astype(np.float64), g.astype(np.float64)
    k = np.stack([ok.k0(x[i], x, g[i], g, kernel, bandwidth=h, **prm) for i in range(n)])
    terms = k * (w.astype(np.float64) if weighted else 1.0)
    # coordinate sums in FP32, as test_gpu_ksd_total; the terms of a row differ in sign
    assert np.abs(part.sum(0).cpu().numpy() - terms.sum(1)).max() <= 5e-6 * np.abs(terms).sum(1).max()


@pytest.mark.parametrize("n", [1, 513, 4096, 5000])
@pytest.mark.parametrize("adaptive", [0, 1])
def test_temper_by_one_workgroup(n, adaptive):
    """In place, against the split step (whose values test_gpu_smc_split holds): the same below 4096 particles, sums in
    another order above."""
    from mocat_amd import _lib, transport  # noqa: F401
    rs = np.random.default_rng(n)
    lw, lik, alpha = (torch.tensor(t.astype(np.float32), device="cuda") for t in
                      (rs.normal(size=n), 10 * rs.gamma(2.0, size=n), rs.uniform(size=(2, n))))
    split, one = torch.empty_like(lw), lw.clone()
    out = [torch.empty(8, dtype=torch.float64, device="cuda") for _ in range(2)]
    nb = _lib.c_i64(0)
    _lib.call("mocat_smc_temper_workspace_bytes", _lib.ctypes.byref(nb))
    ws = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    args = (_lib.ptr(lik), n, 0.1, float(n), 0.2, 1.0, 1e-5, 1000, adaptive, 0.3, _lib.ptr(alpha), 2, math.log(0.1), 1.0,
            0.651)
    _lib.call("mocat_smc_temper_split", _lib.ptr(lw), *args, _lib.ptr(split), _lib.ptr(out[0]), _lib.ptr(ws), nb.value,
              1 << 22, _lib.stream_handle())
    _lib.call("mocat_smc_temper", _lib.ptr(one), *args, _lib.ptr(one), _lib.ptr(out[1]), _lib.stream_handle())
    if n < 4096:
        assert torch.equal(out[0], out[1]) and torch.equal(split, one)
    else:  # FP64 sums of 5000 positive terms; a search step is a quotient of differences of their logarithms
        np.testing.assert_allclose(out[1].cpu().numpy(), out[0].cpu().numpy(), rtol=1e-8, atol=1e-8)
        np.testing.assert_allclose(one.cpu().numpy(), split.cpu().numpy(), rtol=1e-6, atol=1e-6)
