"""Chunked filters around the sizes where the chunk totals move from a wave to a workgroup's LDS and to memory: the
same ancestors, weights and statistics as one workgroup per filter, under every launch mode."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [[4097], [64 * 1024, 100], [64 * 1024 + 1, 5000], [1024 * 1024], [1024 * 1024 + 1, 70000]])
@pytest.mark.parametrize("method", ["systematic", "multinomial"])
@pytest.mark.parametrize("launch", ["stream", "graph", "persistent"])
def test_chunk_offsets(ns, method, launch):
    import mocat_amd as m
    T = 3
    rs = np.random.default_rng(7)
    models = [m.ssm.StochasticVolatility(1, 0.0, 1.0, 0.95, 0.04, 0.6) for _ in ns]
    ys = [rs.normal(size=(T, 1)).astype(np.float32) for _ in ns]
    keys = list(m.random.split(m.random.PRNGKey(5), len(ns)))
    run = lambda sched: m.ssm.run_particle_filters(models, ys, keys, ns, 1.0, method, store=True, schedule=sched)
    one = run({"large_n": 1 << 40, "launch": "stream"})
    for _ in range(2):
        for a, b in zip(one, run({"large_n": 1, "launch": launch})):
            assert torch.equal(a.ancestors, b.ancestors)
            assert torch.equal(a.value, b.value) and torch.equal(a.log_weight, b.log_weight)
            np.testing.assert_allclose(a.ess.cpu().numpy(), b.ess.cpu().numpy(), rtol=1e-6)
            np.testing.assert_allclose(a.log_likelihood.item(), b.log_likelihood.item(), rtol=1e-10)


@pytest.mark.parametrize("count", [89, 90])  # either side of the work up to which the steps take one launch
def test_many_small_filters(count):
    import mocat_amd as m
    model = m.ssm.StochasticVolatility(1, 0.0, 1.0, 0.95, 0.04, 0.6)
    y = np.random.default_rng(3).normal(size=(3, 1)).astype(np.float32)
    keys, ns = list(m.random.split(m.random.PRNGKey(8), count)), [4096] * count
    run = lambda n: m.ssm.run_particle_filters([model] * count, [y] * count, keys, ns, 1.0, "systematic", store=True, large_n=n)
    for a, b in zip(run(1 << 40), run(1)):
        assert torch.equal(a.ancestors, b.ancestors)
        assert torch.equal(a.value, b.value) and torch.equal(a.log_weight, b.log_weight)
