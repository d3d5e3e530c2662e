"""Batches in which the settings leave the forward kernel of some events open and fix
that of others (a class set by hand, the k-streaming kernel, a spacing that several
workgroups do not take): the others keep their kernel, and the open ones go to
several workgroups where that is the faster way for the whole batch."""
import numpy as np
import pytest

import adtomo_hip as A
from adtomo_hip import ops
from test_forward_forms import MODES, case, check, dev

BIG, SMALL = (70, 66, 33), (24, 20, 12)


@pytest.fixture
def settings(tmp_path):
    saved = str(tmp_path / "tune.json")
    A.save_tune(saved)
    for d in ("float64", "float32"):
        A.clear_tune_classes(d)
        A.set_tune(d, diag_max_l=1 << 30, fwd_segs=0, adj_algo=0)
    yield
    A.load_tune(saved)


@pytest.mark.parametrize("mode", MODES, ids=["f64", "f32", "mixed"])
@pytest.mark.parametrize("fixed, form", [({"fwd_segs": 4}, "one"), ({"diag_max_l": 0}, "stream")])
def test_a_fixed_class_keeps_only_its_own_events(settings, mode, fixed, form):
    dtype, mix = mode
    shapes = [BIG, SMALL, BIG] * 20
    assert set(ops.selftest_forward_forms(shapes, dtype, compute_f64=mix)) <= {"team", "wide"}
    A.set_tune_class(SMALL, dtype, **fixed)
    got = ops.selftest_forward_forms(shapes, dtype, compute_f64=mix)
    assert set(got[1::3]) == {form}
    assert set(got[0::3] + got[2::3]) <= {"team", "wide"}


def test_an_event_that_several_workgroups_do_not_take(settings):
    got = ops.selftest_forward_forms([BIG, SMALL, BIG, SMALL, BIG], hs=[0.5, np.nan, 0.5, 1e100, 0.5])
    assert got == ["team", "one", "team", "one", "team"]


def test_all_stay_where_a_fixed_event_would_be_waited_for_twice(settings):
    # one workgroup on 128x128x64 takes 9 ms an iteration, the others less than 5
    # beside it on their own
    shapes = [(128, 128, 64)] + [(64, 64, 32)] * 200
    A.set_tune_class((128, 128, 64), "float64", fwd_segs=8)
    assert set(ops.selftest_forward_forms(shapes)) == {"one"}


@pytest.mark.gpu
@pytest.mark.parametrize("fixed, form", [({"fwd_segs": 4}, "one"), ({"diag_max_l": 0}, "stream")])
@pytest.mark.parametrize("mode", MODES, ids=["f64", "f32", "mixed"])
def test_mixed_batch_bit_exact(settings, mode, fixed, form):
    A.set_tune_class(SMALL, mode[0], **fixed)
    ev = [case(s, mode) for s in (BIG, SMALL, (40, 41, 8))] * 7
    refs = [solve(u0) for u0, _, solve in ev[:3]] * 7
    n = len(ev)
    u0s, fs = [dev(u0) for u0, _, _ in ev], [dev(f) for _, f, _ in ev]
    for kernels in (None, "team", "wide"):
        res = ops.selftest_forward(u0s, fs, [0.5] * n, [1e-3] * n, form=kernels, compute_f64=mode[1])
        assert set(res["form"][1::3]) == {form}
        assert set(res["form"][0::3] + res["form"][2::3]) <= ({kernels} if kernels else {"team", "wide"})
        assert res["left"] == [0] * n
        check(res, refs)
    G = A.EikonalGraph(u0s, fs, [0.5] * n, [1e-3] * n, compute_f64=mode[1])
    for _ in range(3):
        G.launch()
        check({"u": G.us, "info": G.infos()}, refs)
    G.close()
