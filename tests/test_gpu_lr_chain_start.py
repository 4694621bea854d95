"""What a sampler starts from on the logistic-regression scenario: the potential and gradient with the sums over rows in
the order of the fused iterations, at sizes where a call of evaluate splits the rows over workgroups."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scenario(rows, d, precision):
    import mocat_amd as m
    g = torch.Generator(device="cuda").manual_seed(rows + d)
    X = torch.randn((rows, d), device="cuda", generator=g)
    y = (torch.rand(rows, device="cuda", generator=g) < 0.5).float()
    return g, m.LogisticRegression(X, y, precision=precision)


@pytest.mark.parametrize("rows,d,precision", [(1505, 65, "bf16x3"), (3041, 64, "bf16x3"), (20007, 100, "bf16x3"),
                                              (193, 50, "fp32"), (2049, 100, "fp32")])
@pytest.mark.parametrize("points", [1, 40, 300])
def test_samplers_take_the_unsplit_evaluation(rows, d, precision, points):
    import mocat_amd as m
    from mocat_amd import _lib, mcmc
    g, sc = _scenario(rows, d, precision)
    x = 0.3 * torch.randn((points, d), device="cuda", generator=g)
    one = [torch.empty(points, device="cuda"), torch.empty(points, device="cuda"), torch.empty_like(x),
           torch.empty_like(x)]
    _lib.call("mocat_lr_potential_grad", *sc.kernel_args(), 0.7, _lib.ptr(x), points, *[_lib.ptr(t) for t in one],
              _lib.stream_handle())
    got = mcmc.evaluate(sc, x, 0.7)  # the potentials of every sampler
    assert all(torch.equal(a, b) for a, b in zip(got, one))
    sc.temperature = 0.7
    s = m.Underdamped(stepsize=0.01, leapfrog_steps=2)
    st, _ = s.startup(sc, 3, m.cdict(value=x.clone()), m.cdict(random_key=m.random.PRNGKey(1)), n_chains=points)
    assert torch.equal(st.grad_potential, one[2] + 0.7 * one[3])
    assert torch.equal(st.potential, one[0] + 0.7 * one[1])


@pytest.mark.parametrize("rows,d,precision", [(3041, 64, "bf16x3"), (1505, 65, "bf16x3"), (257, 33, "fp32")])
def test_a_chain_alone_is_the_same_chain_in_a_batch(rows, d, precision):
    """4097 chains are past the sizes that evaluate splits; one chain is within them."""
    import mocat_amd as m
    g, sc = _scenario(rows, d, precision)
    x = 0.3 * torch.randn((4097, d), device="cuda", generator=g)
    key = m.random.PRNGKey(5)
    sampler = lambda: m.Underdamped(stepsize=0.02, leapfrog_steps=5)
    batch = m.run(sc, sampler(), 4, key, initial_state=m.cdict(value=x.clone()), n_chains=4097,
                  correction=m.Uncorrected)
    keys = m.random.split(key, 4097)
    for c in (0, 2048, 4096):
        alone = m.run(sc, sampler(), 4, keys[c].contiguous(), initial_state=m.cdict(value=x[c:c + 1].clone()),
                      correction=m.Uncorrected)
        assert torch.equal(alone.value, batch.value[:, c]) and torch.equal(alone.potential, batch.potential[:, c])
        assert torch.equal(alone.final_state.grad_potential[0], batch.final_state.grad_potential[c])
