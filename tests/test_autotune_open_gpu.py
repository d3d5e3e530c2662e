"""adt_autotune on a batch that takes one workgroup per event says nothing of several:
the class stays open, so that a launch of one of its events still takes several, and
the batch its tuned kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import adtomo_hip as A  # noqa: E402
from adtomo_hip import ops  # noqa: E402
from test_forward_forms import MODES, case, dev  # noqa: E402


def test_class_of_a_full_batch_stays_open(tmp_path):
    import torch
    shape, n = (60, 128, 64), 250
    saved = str(tmp_path / "tune.json")
    A.save_tune(saved)
    u0, f, solve = case(shape, MODES[0])
    u0, f = dev(u0), dev(f)
    try:
        A.clear_tune_classes("float64")
        A.set_tune("float64", diag_max_l=1 << 30, fwd_segs=0, adj_algo=0)
        assert set(ops.selftest_forward_forms([shape] * n)) == {"one"}
        A.autotune([u0] * n, [f] * n, [0.5] * n, [1e-3] * n, reps=1)
        (c,) = A.tune_classes("float64")
        print("class:", c, flush=True)
        want = "team" if c["diag_max_l"] else "stream"  # k-streaming fixes the class
        assert ops.selftest_forward_forms([shape]) == [want]
        assert set(ops.selftest_forward_forms([shape] * n)) == {"one" if c["diag_max_l"] else "stream"}
        # the setting survives a file
        A.save_tune(saved + "2")
        A.clear_tune_classes("float64")
        A.load_tune(saved + "2")
        assert ops.selftest_forward_forms([shape]) == [want]
        assert c["diag_max_l"] == 1 << 30  # (the diagonal forward, by a factor)
    finally:
        A.load_tune(saved)
    ref = solve(u0.cpu().numpy())[0]
    u = A.eikonal3d(u0, f, 0.5, *shape, 1e-3, False)
    assert np.array_equal(u.cpu().numpy().view(np.uint64), ref.view(np.uint64))
    torch.cuda.synchronize()
