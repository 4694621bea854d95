"""FP32 logistic regression with the rows of X split over workgroups: the error against the FP64 engine is that of one
workgroup per tile, where the split and its parts begin, with ragged last blocks and few to many points."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [192, 193, 257, 2049, 6001])
@pytest.mark.parametrize("d", [2, 64, 65, 128])
@pytest.mark.parametrize("points", [1, 33, 4096, 4097])
def test_split_rows_fp32(rows, d, points):
    import mocat_amd as m
    from mocat_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(rows + d)
    X = torch.randn((rows, d), device="cuda", generator=g)
    y = (torch.rand(rows, device="cuda", generator=g) < 0.5).float()
    x = 0.3 * torch.randn((points, d), device="cuda", generator=g)
    sc = m.LogisticRegression(X, y, precision="fp32")
    got = sc.evaluate(x)
    want = m.LogisticRegression(X, y, precision="fp64").evaluate(x)
    one = [torch.empty_like(t) for t in got]
    _lib.call("mocat_lr_potential_grad", *sc.kernel_args(), 1.0, _lib.ptr(x), points, *[_lib.ptr(t) for t in one],
              _lib.stream_handle())
    assert torch.equal(got[0], one[0]) and torch.equal(got[2], one[2])  # the prior's
    for k in (1, 3):
        scale = torch.linalg.norm(want[k].double())
        err, ref = (float(torch.linalg.norm(t.double() - want[k].double()) / scale) for t in (got[k], one[k]))
        # both are FP32 sums of at most 6001 terms, one in order, one in parts: neither beats the other by much
        assert err <= 1.5 * ref + 2e-7 and err < 1e-5
    nb = _lib.c_i64(0)
    _lib.call("mocat_lr_eval_workspace_bytes", rows, d, 0, points, _lib.ctypes.byref(nb))
    assert (nb.value > 0) == (rows > 192 and points <= 4096)
