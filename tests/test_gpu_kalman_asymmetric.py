"""Kalman filter and smoother on covariances that are not symmetric (only the kernels use P = P^T) against the formulas,
which take them as they are; symmetric up to rounding they stay with the kernels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,at", [(2, 0), (4, 2), (8, 3)])
@pytest.mark.parametrize("skew", [0.0, 1e-15, 1e-7, 0.1])
def test_smoother_of_asymmetric_covariances(d, at, skew):
    import mocat_amd as m
    rs = np.random.default_rng(d)
    T = 5
    A = 0.9 * np.linalg.qr(rs.standard_normal((d, d)))[0]
    Q = 0.2 * (np.eye(d) + 0.3)
    md = m.ssm.TimeHomogenousLinearGaussian(np.zeros(d), np.eye(d), A, Q, np.eye(d), np.eye(d))
    f, F = rs.standard_normal((T, d)), np.tile(np.eye(d) + 0.3, (T, 1, 1))
    F[at, 0, d - 1] += skew
    F[at, d - 1, 0] -= skew
    got = m.ssm.run_kalman_smoother_for_marginals(md, np.zeros((T, d)), filter_output=(torch.tensor(f, device="cuda"),
                                                                                       torch.tensor(F, device="cuda")))
    mean, cov = f[-1], F[-1]
    for k in range(T - 2, -1, -1):
        J = F[k] @ A.T @ np.linalg.inv(A @ F[k] @ A.T + Q)
        mean, cov = f[k] + J @ (mean - A @ f[k]), F[k] + J @ (cov - A @ F[k] @ A.T - Q) @ J.T
        np.testing.assert_allclose(got[0][k].cpu().numpy(), mean, rtol=1e-10, atol=1e-11)
        np.testing.assert_allclose(got[1][k].cpu().numpy(), cov, rtol=1e-10, atol=1e-11)


@pytest.mark.parametrize("name", ["initial_covariance", "transition_covariance"])
@pytest.mark.parametrize("d,dy", [(2, 2), (4, 1), (3, 8)])
@pytest.mark.parametrize("skew", [0.0, 1e-15, 1e-7, 0.1])
def test_asymmetric_models(d, dy, name, skew):
    import mocat_amd as m
    rs = np.random.default_rng(d)
    A = 0.9 * np.linalg.qr(rs.standard_normal((d, d)))[0]
    H, R = rs.standard_normal((dy, d)), 0.5 * np.eye(dy)
    md = m.ssm.TimeHomogenousLinearGaussian(np.zeros(d), np.eye(d) + 0.3, A, 0.2 * (np.eye(d) + 0.3), H, R)
    cov = getattr(md, name).copy()
    cov[0, d - 1] += skew
    cov[d - 1, 0] -= skew
    setattr(md, name, cov)
    y = rs.standard_normal((4, dy))
    out = m.ssm.run_kalman_filter_for_marginals(md, y)
    mean, P, Q = md.initial_mean, md.initial_covariance, md.transition_covariance
    means, covs = [], []
    for k in range(4):
        if k:
            mean, P = A @ mean, A @ P @ A.T + Q
        L = np.linalg.cholesky(H @ P @ H.T + R)  # of the lower triangle
        K = P @ H.T @ np.linalg.inv(L @ L.T)
        mean, P = mean + K @ (y[k] - H @ mean), P - K @ H @ P
        means.append(mean)
        covs.append(P)
    np.testing.assert_allclose(out[0].cpu().numpy(), np.array(means), rtol=1e-10, atol=1e-11)
    np.testing.assert_allclose(out[1].cpu().numpy(), np.array(covs), rtol=1e-10, atol=1e-11)
    # the smoother alone, on symmetric filter covariances
    f, F = rs.standard_normal((4, d)), np.tile(np.eye(d) + 0.3, (4, 1, 1))
    got = m.ssm.run_kalman_smoother_for_marginals(md, y, filter_output=(torch.tensor(f, device="cuda"),
                                                                        torch.tensor(F, device="cuda")))
    J = F[2] @ A.T @ np.linalg.inv(A @ F[2] @ A.T + Q)
    np.testing.assert_allclose(got[0][2].cpu().numpy(), f[2] + J @ (f[3] - A @ f[2]), rtol=1e-10, atol=1e-11)
