"""Gumbel-max draws by whole wavefronts: rows at the edges of the 64-lane blocks, odd and even row counts
(paired rows share threefry blocks), logits far apart, equal and -inf, against the oracle's FP64 scores."""
import numpy as np
import pytest
import torch

from oracle import rng as orng

pytestmark = pytest.mark.gpu

# scores are formed in FP32: a few ulp of |score| (at most 2e-5 here) can exchange the best two
TIE = 2e-5


@pytest.mark.parametrize("kind", ["normal", "spread", "equal", "holes"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 1000])
@pytest.mark.parametrize("n_out", [1, 2, 7, 64])
def test_categorical_rows(n, n_out, kind):
    import mocat_amd as m
    rs = np.random.default_rng(1000 * n + n_out)
    lw = {"normal": rs.standard_normal(n), "spread": 30.0 * rs.standard_normal(n), "equal": np.zeros(n),
          "holes": np.where(rs.uniform(size=n) < 0.7, -np.inf, rs.standard_normal(n))}[kind].astype(np.float32)
    lw[rs.integers(0, n)] = 1.0
    got = m.ssm.categorical(m.random.PRNGKey(n), torch.tensor(lw, device="cuda"), n_out).cpu().numpy()
    with np.errstate(invalid="ignore"):  # -inf scores: -inf - (-inf) margins
        want, margin = orng.categorical_margin(orng.PRNGKey(n), lw, n_out)
    clear = ~(margin <= TIE)
    np.testing.assert_array_equal(got[clear], want[clear])
    assert clear.sum() >= n_out - 1


@pytest.mark.parametrize("n", [1, 2, 63, 64, 255, 256, 1025])
def test_categorical_filter_paths_agree(n):
    """The same ancestors and weights whichever path the filter takes (one workgroup or the whole GPU)."""
    import mocat_amd as m
    from mocat_amd import datasets
    model, y, _ = datasets.lgssm_config(3, 2, 6)
    y = y.cpu().numpy()
    run = lambda large_n: m.ssm.run_particle_filters([model], [y], [m.random.PRNGKey(n)], [n], 1.0, "categorical",
                                                     store=True, large_n=large_n)[0]
    one, spread = run(1 << 30), run(1)
    assert torch.equal(one.ancestors, spread.ancestors)
    assert torch.equal(one.value, spread.value) and torch.equal(one.log_weight, spread.log_weight)
    np.testing.assert_allclose(one.log_likelihood.item(), spread.log_likelihood.item(), rtol=1e-12)
