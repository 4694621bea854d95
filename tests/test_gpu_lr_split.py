"""Logistic regression with the rows of X split over workgroups: the error against the FP64 engine is that of one
workgroup per tile, at the row counts where the split and its parts begin, ragged last blocks, and few to many points."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1504, 1505, 3040, 3041, 20007])
@pytest.mark.parametrize("d", [3, 64, 65, 128])
@pytest.mark.parametrize("points", [1, 33, 257, 4096])
def test_split_rows(rows, d, points):
    import mocat_amd as m
    from mocat_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(rows + d)
    X = torch.randn((rows, d), device="cuda", generator=g)
    y = (torch.rand(rows, device="cuda", generator=g) < 0.5).float()
    x = 0.3 * torch.randn((points, d), device="cuda", generator=g)
    sc = m.LogisticRegression(X, y)
    got = [t.double() for t in sc.evaluate(x)]
    want = [t.double() for t in m.LogisticRegression(X, y, precision="fp64").evaluate(x)]
    one = [torch.empty_like(t, dtype=torch.float32) for t in got]
    _lib.call("mocat_lr_potential_grad", *sc.kernel_args(), 1.0, _lib.ptr(x), points, *[_lib.ptr(t) for t in one],
              _lib.stream_handle())
    assert torch.equal(got[0], one[0].double()) and torch.equal(got[2], one[2].double())  # the prior's
    for k in (1, 3):
        scale = torch.linalg.norm(want[k])
        err, ref = (float(torch.linalg.norm(t.double() - want[k]) / scale) for t in (got[k], one[k]))
        # the split products' error is common to both; the order of at most 20007 FP32 additions is not
        assert err <= 1.5 * ref + 1e-6 and err < 1e-4
    nb = _lib.c_i64(0)
    _lib.call("mocat_lr_eval_workspace_bytes", rows, d, 1, points, _lib.ctypes.byref(nb))
    blocks = -(-rows // 32)
    assert (nb.value > 0) == (blocks >= (96 if d <= 64 else 48))
