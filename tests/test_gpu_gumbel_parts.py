"""Categorical resampling with the rows split over the waves of a workgroup: the same ancestors as one workgroup per
filter, at the sizes where the number of waves changes, odd and even (paired) rows, and with rows of equal weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [[1], [64], [65, 2], [1535], [1536], [1537], [4095], [4096], [1024, 3000], [300] * 9])
@pytest.mark.parametrize("scale", [1.0, 0.0])
def test_parts_agree(ns, scale):
    import mocat_amd as m
    from mocat_amd import datasets
    model, y, _ = datasets.lgssm_config(3, 2, 4)
    y = y.cpu().numpy()
    keys = list(m.random.split(m.random.PRNGKey(sum(ns)), len(ns)))
    run = lambda large_n: m.ssm.run_particle_filters([model] * len(ns), [y * scale] * len(ns), keys, ns, 1.0, "categorical",
                                                     store=True, large_n=large_n)
    for one, step in zip(run(1 << 30), run(1)):
        assert torch.equal(one.ancestors, step.ancestors)
        assert torch.equal(one.value, step.value) and torch.equal(one.log_weight, step.log_weight)
