"""Schedule records are used only for the kernels, the device and the resampling rate that they were timed with."""
import hashlib
import json

import numpy as np

from mocat_amd.ssm import schedule as sched


class _Model:
    kernel_model, dim, dim_obs = 1, 1, 1


def test_a_record_of_other_kernels_devices_or_thresholds_is_tuned_again(tmp_path, monkeypatch):
    ys, ns = [np.zeros((5, 1)), np.zeros((9, 1))], [300, 700]
    shapes = np.asarray(sorted((n, len(y)) for n, y in zip(ns, ys)), np.int64)
    before = f"1-1-1-default-systematic-g0-s0-{hashlib.sha1(shapes.tobytes()).hexdigest()[:16]}"  # neither was named
    path = tmp_path / "sched.json"
    path.write_text(json.dumps({before: {"large_n": 8192, "launch": "graph"}}))
    monkeypatch.setenv("MOCAT_AMD_SCHEDULE_CACHE", str(path))
    monkeypatch.setattr(sched, "_MEMO", {})
    monkeypatch.setattr(sched.torch.cuda, "synchronize", lambda: None)
    calls = []

    def tuned(ess):
        calls.clear()
        sched.choose(sched.signature([_Model()] * 2, ys, ns, "systematic", False, False, None, ess), calls.append)
        return bool(calls)

    assert tuned(1.0) and not tuned(1.0)
    assert tuned(0.5) and not tuned(0.5)
    monkeypatch.setattr(sched, "KERNEL_VERSION", sched.KERNEL_VERSION + 1)
    assert tuned(1.0) and not tuned(1.0)
    monkeypatch.setattr(sched, "_device", lambda: "another device")
    assert tuned(1.0) and not tuned(1.0)
