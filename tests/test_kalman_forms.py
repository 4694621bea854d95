"""Which calls of the Kalman entries reach the kernels: models whose shapes do not fit (d, dy) take the torch
operations, which raise or broadcast. On the CPU, with every kernel call refused."""
import numpy as np
import pytest
import torch

from mocat_amd.ssm import TimeHomogenousLinearGaussian, filtering


class _Kernel(Exception):
    pass


@pytest.fixture(autouse=True)
def no_kernels(monkeypatch):
    def call(*args):
        raise _Kernel
    monkeypatch.setattr(filtering._lib, "call", call)
    monkeypatch.setattr(filtering._lib, "ptr", lambda t: None)
    monkeypatch.setattr(filtering._lib, "stream_handle", lambda: None)
    monkeypatch.setattr(filtering.mr, "default_device", lambda: torch.device("cpu"))


def _model(d, dy, **other):
    rs = np.random.default_rng(d + dy)
    spd = lambda k, s: s * (np.eye(k) + 0.3 * np.ones((k, k)))
    md = TimeHomogenousLinearGaussian(rs.standard_normal(d), spd(d, 1.0),
                                      0.9 * np.linalg.qr(rs.standard_normal((d, d)))[0], spd(d, 0.2),
                                      rs.standard_normal((dy, d)), spd(dy, 0.5))
    for k, v in other.items():
        setattr(md, k, v)
    return md


@pytest.mark.parametrize("d,dy", [(4, 3), (1, 1), (8, 8), (2, 5)])
def test_fitting_shapes_reach_the_kernels(d, dy):
    md, y = _model(d, dy), np.zeros((3, dy))
    with pytest.raises(_Kernel):
        filtering.run_kalman_filter_for_marginals(md, y)
    with pytest.raises(_Kernel):
        filtering.run_kalman_smoother_for_marginals_and_lag_ones(
            md, y, filter_output=(torch.zeros(3, d), torch.eye(d).expand(3, d, d)))


# a mean shorter and longer than d: packed, the observations behind it would move and the last be read past the end
@pytest.mark.parametrize("other", [
    {"initial_mean": np.zeros(1)}, {"initial_mean": np.zeros(6)}, {"initial_covariance": np.eye(3)},
    {"transition_covariance": np.eye(2)}, {"transition_covariance": np.eye(5)}, {"likelihood_covariance": np.eye(2)},
    {"transition_matrix": np.ones((4, 2))}, {"transition_matrix": np.ones((5, 4))},
    {"likelihood_matrix": np.ones((3, 3))}])
def test_mismatched_filter_raises(other):
    with pytest.raises(RuntimeError, match="size|shapes"):
        filtering.run_kalman_filter_for_marginals(_model(4, 3, **other), np.zeros((2, 3)))


@pytest.mark.parametrize("shape", [(0,), (0, 3), (3, 0)])
def test_no_observations_raise(shape):
    with pytest.raises(RuntimeError, match="reshape tensor of 0|size"):
        filtering.run_kalman_filter_for_marginals(_model(4, 3), np.zeros(shape))


def test_broadcast_covariances():
    y = np.random.default_rng(0).standard_normal((3, 2))
    md = _model(3, 2, transition_covariance=np.full((1, 1), 0.2), likelihood_covariance=np.full((1, 1), 0.5))
    means, covs = filtering.run_kalman_filter_for_marginals(md, y)
    A, H, m, P = md.transition_matrix, md.likelihood_matrix, md.initial_mean, md.initial_covariance
    for k in range(3):
        if k:
            m, P = A @ m, A @ P @ A.T + 0.2
        K = P @ H.T @ np.linalg.inv(H @ P @ H.T + 0.5)
        m, P = m + K @ (y[k] - H @ m), P - K @ H @ P
        np.testing.assert_allclose(means[k], m, rtol=1e-10, atol=1e-11)
        np.testing.assert_allclose(covs[k], P, rtol=1e-10, atol=1e-11)


def test_mismatched_smoother():
    f = (torch.zeros(3, 3, dtype=torch.float64), torch.eye(3, dtype=torch.float64).expand(3, 3, 3))
    smooth = lambda **other: filtering.run_kalman_smoother_for_marginals_and_lag_ones(_model(3, 2, **other),
                                                                                      np.zeros((3, 2)), filter_output=f)
    with pytest.raises(RuntimeError, match="size|shapes"):
        smooth(transition_covariance=np.eye(2))
    with pytest.raises(RuntimeError, match="size|shapes"):
        smooth(transition_matrix=np.ones((3, 2)))
    one = smooth(transition_covariance=np.full((1, 1), 0.2))
    fm, fc = f[0][0], f[1][0]
    A = torch.as_tensor(_model(3, 2).transition_matrix)
    J = fc @ A.T @ torch.linalg.inv(A @ fc @ A.T + 0.2)
    assert torch.allclose(one[1][1], fc + J @ (f[1][2] - A @ fc @ A.T - 0.2) @ J.T, rtol=1e-12, atol=1e-13)


def _smooth(md, means, covs):
    return filtering.run_kalman_smoother_for_marginals_and_lag_ones(md, np.zeros((3, 2)), filter_output=(means, covs))


def test_smoother_is_differentiable_in_the_filter():
    md = _model(2, 2)
    g = torch.Generator().manual_seed(0)
    means = torch.randn((3, 2), dtype=torch.float64, generator=g)
    covs = torch.eye(2, dtype=torch.float64).expand(3, 2, 2).contiguous()
    with pytest.raises(_Kernel):
        _smooth(md, means, covs)
    f = lambda m, c: sum(t.sum() for t in _smooth(md, m, c))
    inputs = (means.clone().requires_grad_(), covs.clone().requires_grad_())
    assert torch.autograd.gradcheck(f, inputs, check_forward_ad=True)
    with torch.no_grad(), pytest.raises(_Kernel):  # no graph asked for
        _smooth(md, *inputs)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(means, torch.ones_like(means))
        assert torch.autograd.forward_ad.unpack_dual(_smooth(md, dual, covs)[0]).tangent is not None


def test_smoother_under_vmap_and_tracing():
    md = _model(2, 2)
    means = torch.randn((4, 3, 2), dtype=torch.float64, generator=torch.Generator().manual_seed(1))
    covs = torch.eye(2, dtype=torch.float64).expand(3, 2, 2).contiguous()
    many = torch.func.vmap(lambda m: _smooth(md, m, covs)[0])(means)
    for k in range(4):
        one = _smooth(md, means[k].requires_grad_(), covs)[0]
        assert torch.allclose(many[k], one, rtol=1e-12, atol=1e-13)
    from torch.fx.experimental.proxy_tensor import make_fx
    traced = make_fx(lambda m: _smooth(md, m, covs)[0])(means[0].detach())
    assert torch.allclose(traced(means[1].detach()), many[1], rtol=1e-12, atol=1e-13)
