"""The 3D adjoint by 8x8x8 tiles with several workgroups per event
(kernels_adjoint_tile.hip) against the CPU oracle: sizes at the edges of a tile,
thin and long boxes, FP64 and FP32, random fields (short cycles between tiles,
many nodes without feeders), fields with no node to solve, batches of events of
different sizes, graph replays.  Each node's result is
the oracle's operations in the oracle's order; the tolerance leaves room for one
rounding in each of a chain of some thousand steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle  # noqa: E402
from adtomo_hip import synth  # noqa: E402


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def case(shape, seed, dt=np.float64, rough=False):
    r = synth.rng(seed)
    f = 1.0 / synth.layered_grf_model(shape, 0.5, std=0.05, corr_km=1.0, seed=seed)
    u0 = synth.point_source_u0(shape, tuple(int(r.integers(0, s)) for s in shape))
    u = r.uniform(1.0, 2.0, size=shape) if rough else oracle.eikonal3d(u0, f, 0.5, 1e-4)[0]
    g = r.normal(size=shape)
    return [a.astype(dt) for a in (g, u, u0, f)]


def check(got, args):
    gu0, gf = (a.cpu().numpy() for a in got)
    dt = gf.dtype.type
    r0, rf, _ = oracle.eikonal3d_grad(*args, 0.5, dtype=dt)
    tol = 4000 * np.finfo(dt).eps
    assert np.array_equal(gu0, r0)
    assert np.abs(gf - rf).max() <= tol * max(np.abs(rf).max(), np.finfo(dt).tiny)


@pytest.mark.parametrize("rough", [False, True])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [
    (2, 2, 2), (8, 8, 8), (9, 8, 7), (7, 17, 16), (16, 9, 33), (2, 3, 200), (150, 2, 5),
    (40, 41, 39)])
def test_tiles_one_event(shape, dt, rough):
    import adtomo_hip as A
    args = case(shape, sum(shape), dt, rough)
    for _ in range(3):
        check(A.eikonal3d_grad(*(dev(a) for a in args), 0.5, *shape), args)


def test_tiles_nothing_to_solve():
    import adtomo_hip as A
    g, u, u0, f = case((20, 9, 11), 3)
    got = A.eikonal3d_grad(dev(g), dev(u0), dev(u0), dev(f), 0.5, 20, 9, 11)
    assert np.array_equal(got[0].cpu().numpy(), g) and not np.abs(got[1].cpu().numpy()).any()
    assert A.ops.last_info["adj_converged"] == 1


def test_tiles_batch_and_graph_replays():
    import torch
    import adtomo_hip as A
    r = synth.rng(8)
    shapes = [tuple(int(x) for x in r.integers(2, 50, size=3)) for _ in range(30)]
    cs = [case(s, 50 + e, rough=e % 3 == 0) for e, s in enumerate(shapes)]
    g, u, u0, f = ([dev(c[q]) for c in cs] for q in range(4))
    n = len(cs)
    res = A.eikonal3d_batched(u0, f, [0.5] * n, [1e-4] * n, grad_us=g, us=u, forward=False)
    for e in range(n):
        check((res["grad_u0"][e], res["grad_f"][e]), cs[e])
    want = [a.clone() for a in res["grad_f"]]
    G = A.EikonalGraph(u0, f, [0.5] * n, [1e-4] * n, grad_us=g, us=u, forward=False)
    for _ in range(4):
        for x in G.grad_fs:
            x.fill_(-1.0)
        G.launch()
        torch.cuda.synchronize()
        assert all(i["adj_converged"] == 1 for i in G.infos())
        assert all(torch.equal(G.grad_fs[e], want[e]) for e in range(n))
    G.close()
