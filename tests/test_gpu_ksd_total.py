"""The pairwise total of the kernel Stein discrepancy (pairs i <= j in 64 x 64 tiles) at tile edges, for both
kernels, the inverse multiquadric's usual and other exponents, and weights, against the FP64 oracle."""
import numpy as np
import pytest
import torch

from oracle import ksd as ok

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d", [(1, 1), (2, 33), (64, 32), (65, 31), (129, 5), (200, 128)])
@pytest.mark.parametrize("kern", ["gaussian", "imq", "imq_other"])
@pytest.mark.parametrize("weighted", [False, True])
def test_total_vs_oracle(n, d, kern, weighted):
    import mocat_amd as m
    rs = np.random.default_rng(3 * n + d)
    x = rs.normal(0.5, 1.2, (n, d)).astype(np.float32)
    g = (0.8 * x + rs.normal(0, 0.3, (n, d))).astype(np.float32)
    lw = rs.normal(0, 1, n).astype(np.float32) if weighted else None
    h = 0.7 * np.sqrt(d)
    prm = dict(bandwidth=h) if kern == "gaussian" else dict(c=1.0, beta=-0.5 if kern == "imq" else -0.75, bandwidth=h)
    kernel = m.kernels.Gaussian(**prm) if kern == "gaussian" else m.kernels.IMQ(**prm)
    got = m.ksd(torch.tensor(x), kernel, grad_potential=torch.tensor(g),
                log_weight=None if lw is None else torch.tensor(lw))
    want = ok.ksd(x, g, "gaussian" if kern == "gaussian" else "imq", log_weight=lw, **prm)
    # coordinate sums in FP32: about sqrt(d) 2^-24 each, a few of them in every pair's value
    assert got == pytest.approx(want, rel=5e-6), (got, want)
