"""The forward with several workgroups per event and eight nodes of k per lane
(the wide form of kernels_team.hip), which the library takes for many events of
unequal size, against the CPU oracle, bit for bit: boxes at the edges of its bands
(64 rows), of a lane's eight nodes and of a slab (32), in FP64, FP32 and FP32
storage with FP64 solves, one event among them with values that the fast solve
does not cover; graph replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle  # noqa: E402
from adtomo_hip import synth  # noqa: E402

SHAPES = [(2, 2, 2), (9, 7, 16), (63, 65, 7), (64, 64, 9), (65, 66, 31), (128, 67, 18),
          (70, 129, 33), (12, 13, 70), (30, 20, 32), (40, 41, 8)]
COPIES = 24


def dev(a, dtype):
    import torch
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=dtype))).to("cuda")


def bits(t, ref):
    a = t.detach().cpu().numpy()
    w = np.uint64 if a.dtype == np.float64 else np.uint32
    return np.array_equal(a.view(w), ref.view(w))


@pytest.mark.parametrize("mode", ["f64", "f32", "mixed"])
def test_wide_forward_bit_exact(mode):
    import torch
    import adtomo_hip as A
    dt = np.float64 if mode == "f64" else np.float32
    u0s, fs, refs = [], [], []
    for s in SHAPES:
        f = 1.0 / synth.layered_grf_model(s, 0.5, std=0.05, corr_km=1.0, seed=sum(s))
        r = synth.rng(sum(s))
        u0 = synth.point_source_u0(s, tuple(int(r.integers(0, x)) for x in s))
        if s == (30, 20, 32):
            u0[1, 1, 1] = np.nan  # left to the diagonal kernel
        if mode == "mixed":
            refs.append(oracle.eikonal3d_m32(u0, f, 0.5, 1e-3))
        else:
            refs.append(oracle.eikonal3d(u0, f, 0.5, 1e-3, dtype=dt))
        u0s.append(u0)
        fs.append(f)
    n = len(SHAPES) * COPIES
    k = len(SHAPES)
    du = [dev(u0s[e % k], dt) for e in range(n)]
    df = [dev(f, dt) for f in fs] * COPIES
    res = A.eikonal3d_batched(du, df, [0.5] * n, [1e-3] * n, compute_f64=mode == "mixed")
    for e in range(n):
        assert res["info"][e]["iterations"] == refs[e % k][1], (e, SHAPES[e % k])
        assert bits(res["u"][e], refs[e % k][0]), (e, SHAPES[e % k])
    if mode != "f64":
        return
    G = A.EikonalGraph(du, df, [0.5] * n, [1e-3] * n)
    for rep in range(3):
        for u in G.us:
            u.fill_(-1.0)
        G.launch()
        torch.cuda.synchronize()
        assert all(bits(G.us[e], refs[e % k][0]) for e in range(n)), rep
    G.close()
