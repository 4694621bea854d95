"""Kalman filter and smoother kernels (FP64) and, beyond their dimensions, the same entry points'
torch path against the textbook recursions: state and observation dimensions equal, unequal (padding) and at the kernels' limit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(d, dy, seed):
    import mocat_amd as m
    rs = np.random.default_rng(seed)
    spd = lambda k, s: s * (np.eye(k) + 0.3 * np.ones((k, k)))
    return m.ssm.TimeHomogenousLinearGaussian(rs.standard_normal(d), spd(d, 1.0),
                                              0.9 * np.linalg.qr(rs.standard_normal((d, d)))[0], spd(d, 0.2),
                                              rs.standard_normal((dy, d)), spd(dy, 0.5))


def _direct(md, y):
    """The textbook recursions in FP64 numpy."""
    A, Q, H, R = md.transition_matrix, md.transition_covariance, md.likelihood_matrix, md.likelihood_covariance
    m, P, ll, ms, Ps = md.initial_mean, md.initial_covariance, 0.0, [], []
    for k, yk in enumerate(y):
        if k:
            m, P = A @ m, A @ P @ A.T + Q
        S, r = H @ P @ H.T + R, yk - H @ m
        K = np.linalg.solve(S, H @ P).T
        ll -= 0.5 * (r @ np.linalg.solve(S, r) + np.linalg.slogdet(S)[1] + len(r) * np.log(2 * np.pi))
        m, P = m + K @ r, P - K @ H @ P
        ms.append(m)
        Ps.append(P)
    sm, sP, lag = [ms[-1]], [Ps[-1]], []
    for k in range(len(y) - 2, -1, -1):
        pred = A @ Ps[k] @ A.T + Q
        J = np.linalg.solve(pred, A @ Ps[k]).T
        lag.append(ms[k] @ sm[-1] + J @ (sP[-1] + (sm[-1] - ms[k + 1]) @ sm[-1]))
        sm.append(ms[k] + J @ (sm[-1] - A @ ms[k]))
        sP.append(Ps[k] + J @ (sP[-1] - pred) @ J.T)
    return map(np.array, (ms, Ps, ll, sm[::-1], sP[::-1], lag[::-1]))


@pytest.mark.parametrize("d,dy", [(1, 1), (2, 1), (1, 3), (3, 3), (4, 4), (5, 2), (3, 6), (7, 7), (8, 8), (8, 3), (9, 2),
                                  (2, 9)])
@pytest.mark.parametrize("T", [1, 2, 65])
def test_filter_and_smoother(d, dy, T):
    import mocat_amd as m
    md = _model(d, dy, 10 * d + dy)
    y = np.random.default_rng(T).standard_normal((T, dy))
    ms, Ps, ll, sm, sP, lag = _direct(md, y)
    out = m.ssm.run_kalman_filter_for_marginals(md, y)
    got = m.ssm.run_kalman_smoother_for_marginals_and_lag_ones(md, y, filter_output=out)
    # FP64 recursions of well-conditioned models: a few hundred roundings of the values' scale
    close = lambda a, b: np.testing.assert_allclose(a.cpu().numpy(), b, rtol=1e-10, atol=1e-11)
    close(out[0], ms)
    close(out[1], Ps)
    close(out.log_likelihood, ll)
    close(got[0], sm)
    close(got[1], sP)
    close(got[2], lag.reshape(T - 1, d, d))


def test_not_positive_definite_raises_as_before():
    import mocat_amd as m
    md = _model(3, 2, 1)
    md.likelihood_covariance = -10.0 * np.eye(2)
    with pytest.raises(torch.linalg.LinAlgError):
        m.ssm.run_kalman_filter_for_marginals(md, np.zeros((4, 2)))
