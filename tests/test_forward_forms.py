"""Which forward kernel runs.  All forms give the same bits by design, so the tests
that compare them with the oracle name the form and check that it solved the events
itself.  On the CPU: the library's choice for the boxes of the other test files.  On
the device: each form on boxes at the edges of bands (64 rows), lanes (2, 4 and 8
nodes of k), slabs (4 lanes) and segments; events whose values the local solve of
several workgroups does not cover; two batches at once on two streams."""
import numpy as np
import pytest

from adtomo_hip import ops, synth
from test_team_wide_gpu import COPIES, SHAPES as WIDE_SHAPES

MODES = [("float64", False), ("float32", False), ("float32", True)]
SHAPES = [(2, 2, 2), (3, 2, 17), (9, 7, 16), (12, 13, 70), (63, 65, 7), (64, 64, 9), (65, 66, 31),
          (70, 129, 33), (128, 67, 18), (20, 200, 5), (40, 41, 8), (30, 20, 32)]


@pytest.mark.parametrize("dtype, mix", MODES)
def test_choice_for_the_boxes_of_other_tests(dtype, mix):
    for s in [(2, 2, 2), (63, 65, 7), (70, 129, 33), (12, 13, 70), (128, 128, 64)]:
        assert ops.selftest_forward_forms([s], dtype, compute_f64=mix) == ["team"]
    assert set(ops.selftest_forward_forms(WIDE_SHAPES * COPIES, dtype, compute_f64=mix)) <= {
        "team", "wide"}
    assert ops.selftest_forward_forms([(16, 16, 16)], dtype, hs=[np.nan]) == ["one"]


def case(shape, mode):
    from oracle import oracle
    dtype, mix = mode
    f = 1.0 / synth.layered_grf_model(shape, 0.5, std=0.05, corr_km=1.0, seed=sum(shape))
    r = synth.rng(sum(shape))
    u0 = synth.point_source_u0(shape, tuple(int(r.integers(0, x)) for x in shape))
    dt = np.float32 if dtype == "float32" else np.float64
    solve = (lambda u: oracle.eikonal3d_m32(u, f, 0.5, 1e-3)) if mix else (
        lambda u: oracle.eikonal3d(u, f, 0.5, 1e-3, dtype=dt))
    return u0.astype(dt), f.astype(dt), solve


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def check(res, refs):
    w = np.uint64 if refs[0][0].dtype == np.float64 else np.uint32
    for e, (u, it, _) in enumerate(refs):
        assert res["info"][e]["iterations"] == it and res["info"][e]["fault"] == 0, e
        assert np.array_equal(res["u"][e].cpu().numpy().view(w), u.view(w)), e


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["one", "team", "wide"])
@pytest.mark.parametrize("mode", MODES, ids=["f64", "f32", "mixed"])
def test_each_form_bit_exact(mode, form):
    ev = [case(s, mode) for s in SHAPES]
    refs = [solve(u0) for u0, _, solve in ev]
    for copies in (1, 9):  # fewer and more events than XCDs hold at a time
        n = len(ev) * copies
        res = ops.selftest_forward([dev(u0) for u0, _, _ in ev] * copies,
                                   [dev(f) for _, f, _ in ev] * copies, [0.5] * n, [1e-3] * n,
                                   form=form, compute_f64=mode[1])
        assert res["form"] == [form] * n
        # (the 2x2x2 model's slowness is 1e-8: against u0 = 1000 discriminants cancel
        # to 0, which the FP64 solve of several workgroups leaves to one)
        tiny = [float(f.max()) < 1e-6 for _, f, _ in ev] * copies
        assert all(k == 0 or (t and k == 1) for k, t in zip(res["left"], tiny))
        check(res, refs * copies)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["team", "wide"])
def test_only_uncovered_values_are_left_to_one_workgroup(form):
    ev = [case(s, MODES[0]) for s in SHAPES]
    ev[4][0][1, 1, 1] = np.nan
    ev[7][0][2, 2, 2] = -0.0
    ev[9][1][2:4, 2:4, 1:3] = np.inf
    from oracle import oracle
    with np.errstate(invalid="ignore"):
        refs = [oracle.eikonal3d(u0, f, 0.5, 1e-3) for u0, f, _ in ev]
    n = len(ev)
    res = ops.selftest_forward([dev(u0) for u0, _, _ in ev], [dev(f) for _, f, _ in ev],
                               [0.5] * n, [1e-3] * n, form=form)
    assert res["left"] == [1 if e in (0, 4, 7, 9) else 0 for e in range(n)]  # 0: see above
    for e in range(n):
        assert np.array_equal(res["u"][e].cpu().numpy(), refs[e][0], equal_nan=True), e


@pytest.mark.gpu
def test_batches_on_two_streams_at_once():
    import torch
    import adtomo_hip as A
    ev = [case(s, MODES[0]) for s in SHAPES * 4]
    refs = [solve(u0) for u0, _, solve in ev[:len(SHAPES)]] * 4
    n = len(ev)
    u0s, fs = [dev(u0) for u0, _, _ in ev], [dev(f) for _, f, _ in ev]
    graphs = [A.EikonalGraph(u0s, fs, [0.5] * n, [1e-3] * n) for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in graphs]
    torch.cuda.synchronize()
    for _ in range(3):
        for G in graphs:
            for u in G.us:
                u.fill_(-1.0)
        torch.cuda.synchronize()
        for G, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                G.launch()
                G.launch()
        torch.cuda.synchronize()
        for G in graphs:
            check({"u": G.us, "info": G.infos()}, refs)
    for G in graphs:
        G.close()
