"""The bf16x3 logistic-regression engine at the edges of its padded columns, of its 32-row blocks and of its one- and
two-tile workgroups, against FP64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [1, 31, 32, 33, 50, 63, 64, 65, 96, 100, 127, 128])
@pytest.mark.parametrize("n,C", [(1, 1), (33, 31), (300, 65), (97, 16383), (64, 16384 + 33)])
def test_layouts_vs_fp64(n, C, d):
    import mocat_amd as m
    g = torch.Generator(device="cuda").manual_seed(1000 * d + n)
    X = torch.randn((n, d), generator=g, device="cuda")
    y = (torch.rand((n,), generator=g, device="cuda") < 0.5).float()
    th = torch.randn((C, d), generator=g, device="cuda") / d ** 0.5
    sc = m.LogisticRegression(X, y, prior_variance=10.0)
    pp, lp, gp, gl = sc.evaluate(th)
    X64, t64, y64 = X.double(), th.double(), y.double()
    z = t64 @ X64.T
    soft = torch.nn.functional.softplus(z, threshold=1e9)
    # split products leave 2^-16 of each term (the bound of the package's other bf16x3 checks)
    assert ((lp.double() - (soft - y64 * z).sum(1)).abs() / (soft.sum(1) + 1.0)).max().item() < 2e-5
    want = (torch.sigmoid(z) - y64) @ X64
    assert ((gl.double() - want).abs().max() / (X64.abs().sum(0).max() + 1.0)).item() < 1e-4
    assert torch.equal(gp, 0.1 * th) or (gp - 0.1 * th).abs().max().item() < 1e-7


@pytest.mark.parametrize("d,C", [(37, 40), (53, 70), (101, 33), (100, 16384 + 40), (128, 16384)])
def test_chain_iteration_matches_separate_evaluations(d, C):
    """One uncorrected leapfrog step of every chain equals the step formed from the evaluation entry's gradients."""
    import mocat_amd as m
    g = torch.Generator(device="cuda").manual_seed(d)
    X = torch.randn((130, d), generator=g, device="cuda")
    y = (torch.rand((130,), generator=g, device="cuda") < 0.5).float()
    x = torch.randn((C, d), generator=g, device="cuda") / d ** 0.5
    sc = m.LogisticRegression(X, y, prior_variance=10.0)
    h = 0.05
    s = m.Underdamped(stepsize=h, leapfrog_steps=1, friction=0.0)
    ex = m.cdict(random_key=m.random.PRNGKey(d))
    st, ex = s.startup(sc, 10, m.cdict(value=x.clone()), ex, n_chains=C, correction=m.Uncorrected)
    p0 = torch.randn((C, d), generator=g, device="cuda")
    st.momenta = p0.clone()
    g0 = st.grad_potential.clone()
    s.iterate(sc, st, ex, 1)
    half = -p0 - 0.5 * h * g0  # the iteration negates the momentum first (friction 0: no refresh)
    x1 = x + h * half
    pp, lp, gp, gl = sc.evaluate(x1)
    # FP32 rounding of a few operations; the positions differ by roundings of h p
    assert (st.value - x1).abs().max().item() < 5e-7 * (1 + x1.abs().max().item())
    scale = (X.abs().sum(0).max() + 1.0).item()
    assert (st.grad_potential - (gp + gl)).abs().max().item() < 1e-5 * scale
    assert ((st.potential - (pp + lp)).abs() / (pp + lp).abs()).max().item() < 2e-6
    assert (-st.momenta - (half - 0.5 * h * (gp + gl))).abs().max().item() < 1e-5 * scale
