"""A bounded wait of the forward that runs out leaves the event to another kernel,
whose results are right: adt_info.fault says so (2), so that the time-out is seen, and
only a fault without such results (1) is an error.  Several workgroups are told on
entry that their wait has run out; nothing waits."""
import numpy as np
import pytest

from adtomo_hip import _lib as L
from adtomo_hip import ops
from test_forward_forms import MODES, SHAPES, case, dev


def test_fault_codes_in_python():
    ops._checked({"fault": 0})
    with pytest.warns(UserWarning, match="timed out"):
        ops._checked({"fault": 2})
    with pytest.raises(L.AdtError):
        ops._checked({"fault": 1})


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["team", "wide"])
@pytest.mark.parametrize("mode", MODES, ids=["f64", "f32", "mixed"])
def test_events_left_after_a_time_out_say_so(mode, form):
    ev = [case(s, mode) for s in SHAPES[1:]]  # (2x2x2 is left for its values)
    refs = [solve(u0) for u0, _, solve in ev]
    n = len(ev)
    left = [(0, 2, 1)[e % 3] for e in range(n)]
    with pytest.warns(UserWarning, match="timed out"):
        res = ops.selftest_forward([dev(u0) for u0, _, _ in ev], [dev(f) for _, f, _ in ev],
                                   [0.5] * n, [1e-3] * n, form=form, compute_f64=mode[1], left=left)
    assert res["form"] == [form] * n and res["left"] == left
    assert [i["fault"] for i in res["info"]] == [2 if k == 2 else 0 for k in left]
    w = np.uint64 if mode[0] == "float64" else np.uint32
    for e, (u, it, _) in enumerate(refs):
        assert res["info"][e]["iterations"] == it, e
        assert np.array_equal(res["u"][e].cpu().numpy().view(w), u.view(w)), e
