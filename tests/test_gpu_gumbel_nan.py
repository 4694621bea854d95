"""Gumbel-max draws with NaN scores: a NaN is never better than a number, so a particle whose score is NaN is drawn as if
its log-weight were -inf and hides no other one; a row whose first score is NaN takes index 0."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("holes", [(1,), (2,), (5,), (64,), (1, 64, 65, 130), tuple(range(1, 64)), tuple(range(1, 199)), (199,)])
@pytest.mark.parametrize("n_out", [1, 7, 300])
def test_categorical_nan_is_never_taken(n_out, holes):
    import mocat_amd as m
    lw = np.random.default_rng(n_out).standard_normal(200).astype(np.float32)
    a, b = lw.copy(), lw.copy()
    a[list(holes)], b[list(holes)] = np.nan, -np.inf
    draw = lambda w: m.ssm.categorical(m.random.PRNGKey(n_out), torch.tensor(w, device="cuda"), n_out)
    assert torch.equal(draw(a), draw(b))


@pytest.mark.parametrize("n", [1, 2, 65, 200])
@pytest.mark.parametrize("n_out", [1, 8, 9])
def test_categorical_nan_first(n, n_out):
    import mocat_amd as m
    draw = lambda w: m.ssm.categorical(m.random.PRNGKey(3), torch.tensor(w, device="cuda"), n_out)
    lw = np.zeros(n, np.float32)
    lw[0] = np.nan
    assert not draw(lw).any()
    lw[n // 2:] = np.inf
    lw[0] = np.nan
    assert not draw(lw).any()
    assert not draw(np.full(n, np.nan, np.float32)).any()


@pytest.mark.parametrize("what", ["state", "weight"])
@pytest.mark.parametrize("d", [1, 4, 6])  # 6: no compiled transition
@pytest.mark.parametrize("n,m_count", [(63, 17), (512, 40), (1025, 15), (600, 2050)])
def test_backward_simulation_nan_is_never_taken(n, m_count, d, what):
    """The particles with a NaN state or log-weight against the same ones with log-weight -inf, one wave or four
    per trajectory, with and without prepared bounds."""
    import mocat_amd as m
    from mocat_amd import _lib
    rs = np.random.default_rng(100 * n + d)
    ssm = m.ssm.TimeHomogenousLinearGaussian(np.zeros(d), np.eye(d), 0.9 * np.linalg.qr(rs.standard_normal((d, d)))[0],
                                             0.1 * np.eye(d), np.eye(d), np.eye(d))
    params = torch.as_tensor(ssm.transition_params(), device="cuda").contiguous()
    T = 3
    x, lw = rs.standard_normal((T, n, d)).astype(np.float32), rs.standard_normal((T, n)).astype(np.float32)
    holes = np.unique(np.r_[1, 2, rs.integers(1, n, n // 8)])
    clean = lw.copy()
    clean[:, holes] = -np.inf
    bad_x, bad_lw = x.copy(), lw.copy()
    if what == "state":
        bad_x[:, holes, d - 1] = np.nan
    else:
        bad_lw[:, holes] = np.nan
    keys = m.random.split(m.random.PRNGKey(n + d), T).contiguous()
    last = torch.tensor(rs.standard_normal((m_count, d)), dtype=torch.float32, device="cuda")
    nb = _lib.c_i64(0)
    _lib.call("mocat_ffbsi_workspace_bytes", 0, d, T, n, m_count, _lib.ctypes.byref(nb))
    ws = torch.empty(nb.value, dtype=torch.uint8, device="cuda")

    def run(x, lw):
        x, lw = torch.tensor(x, device="cuda"), torch.tensor(lw, device="cuda")
        anc = torch.zeros((T, m_count), dtype=torch.int32, device="cuda")
        out = torch.empty((T, m_count, d), device="cuda")
        out[T - 1] = last
        _lib.call("mocat_ffbsi_run", 0, d, _lib.ptr(params), _lib.ptr(x), _lib.ptr(lw), T, n, m_count, _lib.ptr(keys),
                  _lib.ptr(ws), nb.value, _lib.ptr(anc), _lib.ptr(out), _lib.stream_handle())
        one = torch.empty(m_count, dtype=torch.int32, device="cuda")
        _lib.call("mocat_ffbsi_step", 0, d, _lib.ptr(params), _lib.ptr(x[1]), _lib.ptr(lw[1]), n, _lib.ptr(out[2]), m_count,
                  _lib.ptr(keys[1]), _lib.ptr(one), _lib.ptr(torch.empty((m_count, d), device="cuda")),
                  _lib.stream_handle())
        assert torch.equal(one, anc[1])
        return anc, out

    (anc, out), (want, want_out) = run(bad_x, bad_lw), run(x, clean)
    assert torch.equal(anc, want) and torch.equal(out, want_out)
