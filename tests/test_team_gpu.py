"""The forward with several workgroups per event (kernels_team.hip) against the
CPU oracle, bit for bit: sizes at the edges of its bands (64 rows), slabs (4
waves of 16 bytes of k) and segments, in FP64, FP32 and FP32 storage with FP64
solves; batches of more events than XCDs with boxes of different sizes; events
whose values the fast solve does not cover among others; graph replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle  # noqa: E402
from adtomo_hip import synth  # noqa: E402


def dev(a, dtype=np.float64):
    import torch
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=dtype))).to("cuda")


def same_bits(t, ref):
    a = t.detach().cpu().numpy()
    w = np.uint64 if a.dtype == np.float64 else np.uint32
    return a.shape == ref.shape and np.array_equal(a.view(w), ref.view(w))


def event(shape, seed):
    f = 1.0 / synth.layered_grf_model(shape, 0.5, std=0.05, corr_km=1.0, seed=seed)
    r = synth.rng(seed)
    return f, synth.point_source_u0(shape, tuple(int(r.integers(0, s)) for s in shape))


@pytest.mark.parametrize("shape", [
    (2, 2, 2), (3, 2, 17), (7, 9, 8), (9, 7, 16), (63, 65, 7), (64, 64, 9), (65, 66, 15),
    (128, 67, 18), (70, 129, 33), (20, 200, 5), (12, 13, 70)])
def test_team_forward_bit_exact(shape):
    import adtomo_hip as A
    f, u0 = event(shape, sum(shape))
    ref, it, err = oracle.eikonal3d(u0, f, 0.5, 1e-4)
    for _ in range(3):
        u = A.eikonal3d(dev(u0), dev(f), 0.5, *shape, 1e-4, False)
        assert A.ops.last_info["iterations"] == it and A.ops.last_info["err"] == err
        assert same_bits(u, ref)
    r32, it32, _ = oracle.eikonal3d(u0, f, 0.5, 1e-4, dtype=np.float32)
    rm, itm, _ = oracle.eikonal3d_m32(u0, f, 0.5, 1e-4)
    for mix, r, k in ((False, r32, it32), (True, rm, itm)):
        res = A.eikonal3d_batched([dev(u0, np.float32)], [dev(f, np.float32)], [0.5], [1e-4],
                                  compute_f64=mix)
        assert res["info"][0]["iterations"] == k and same_bits(res["u"][0], r)


def test_team_batch_of_uneven_events_and_graph_replays():
    import torch
    import adtomo_hip as A
    r = synth.rng(5)
    shapes = [tuple(int(x) for x in (r.integers(5, 80), r.integers(5, 80), r.integers(4, 40)))
              for _ in range(21)]
    ev = [event(s, 100 + e) for e, s in enumerate(shapes)]
    ev[4][1][1, 1, 1] = np.nan            # left to the diagonal kernel
    ev[9][0][2:4, 2:4, 1:3] = 1e-170      # discriminants of 0
    refs = [oracle.eikonal3d(u0, f, 0.5, 1e-3) for f, u0 in ev]
    u0s, fs = [dev(u0) for _, u0 in ev], [dev(f) for f, _ in ev]
    n = len(ev)
    res = A.eikonal3d_batched(u0s, fs, [0.5] * n, [1e-3] * n)
    for e in range(n):
        assert res["info"][e]["iterations"] == refs[e][1], (e, shapes[e])
        assert same_bits(res["u"][e], refs[e][0]), (e, shapes[e])
    G = A.EikonalGraph(u0s, fs, [0.5] * n, [1e-3] * n)
    for rep in range(4):
        for u in G.us:
            u.fill_(-1.0)
        G.launch()
        torch.cuda.synchronize()
        assert [i["iterations"] for i in G.infos()] == [x[1] for x in refs]
        assert all(same_bits(G.us[e], refs[e][0]) for e in range(n)), rep
    G.close()
