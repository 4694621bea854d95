"""The one-launch particle-filter step (calls whose largest chunked filter has at most 4096 particles) at the
edges of its 256-particle chunks and 1024-weight scan tiles, against the one-workgroup kernel."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["lg", "lg_multinomial", "optimal", "sv_grad", "sv_times"])
@pytest.mark.parametrize("ns", [[1], [255, 256, 257], [1023, 2], [1025, 1024], [4095, 300, 4096]])
def test_one_launch_step_matches_one_workgroup(case, ns):
    import mocat_amd as m
    from mocat_amd import datasets
    T = [7, 2, 1][:len(ns)]
    F = len(ns)
    keys = list(m.random.split(m.random.PRNGKey(sum(ns)), F))
    kw = {}
    if case.startswith("sv"):
        models, ys, _ = datasets.sv_batch_config(5, F, 10, 20, 8, 8)
        ys = [y[:t] for y, t in zip(ys, T)]
        if case == "sv_times":
            kw["ts"] = [np.cumsum(np.linspace(0.5, 1.5, t)) for t in T]
        else:
            kw["grad"] = True
    else:
        model, y, _ = datasets.lgssm_config(1, 4, 8)
        models, ys = [model] * F, [y.cpu().numpy()[:t] for t in T]
    if case == "optimal":
        kw["particle_filter"] = m.ssm.OptimalNonLinearGaussianParticleFilter
    method = "multinomial" if case == "lg_multinomial" else "systematic"
    for ess in (1.0, 0.5):
        one, step = [m.ssm.run_particle_filters(models, ys, keys, ns, ess, method, store=True, large_n=large_n, **kw)
                     for large_n in (1 << 30, 1)]
        for a, b in zip(one, step):
            assert torch.equal(a.ancestors, b.ancestors)
            assert torch.equal(a.value, b.value) and torch.equal(a.log_weight, b.log_weight)
            assert torch.equal(a.final_value, b.final_value)
            # the FP64 sums of the weights are taken in another order: 4096 terms, n eps
            np.testing.assert_allclose(b.log_likelihood.item(), a.log_likelihood.item(), rtol=1e-12, atol=1e-12)
            np.testing.assert_allclose(b.ess.cpu(), a.ess.cpu(), rtol=2e-7)
            if "grad" in kw:
                np.testing.assert_allclose(b.log_likelihood_grad.cpu(), a.log_likelihood_grad.cpu(), rtol=1e-9, atol=1e-9)
