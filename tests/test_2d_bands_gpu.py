"""The 2D forward by bands of rows and the 2D adjoint with its working values in
LDS (kernels_2d.hip) against the CPU oracle: sizes at the edges of a band (64
rows), of the LDS (values, multipliers, codes) and of the workgroup (8 and 16
bands), both orders of the axes, a source at a corner, slowness that the fast
solve does not cover, levels longer than the LDS queue.  Forward: bit for bit.
Adjoint: the kernel's operations are the
oracle's in its order, in the oracle's precision; the tolerance leaves room for
one rounding in each of a chain of some thousand steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle  # noqa: E402
from adtomo_hip import synth  # noqa: E402


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def same_bits(t, ref):
    a = t.detach().cpu().numpy()
    w = np.uint64 if a.dtype == np.float64 else np.uint32
    return a.shape == ref.shape and np.array_equal(a.view(w), ref.view(w))


def check(f, sx, sy, h, dt, seed=0):
    import adtomo_hip as A
    f = f.astype(dt)
    ref, it, err, _ = oracle.eikonal2d(f, sx, sy, h, dtype=dt)
    u = A.eikonal(dev(f), sx, sy, h)
    assert same_bits(u, ref)
    assert A.ops.last_info["iterations"] == it and A.ops.last_info["err"] == err
    check_adjoint(ref, f, sx, sy, h, seed)


def check_adjoint(u, f, sx, sy, h, seed=0):
    import adtomo_hip as A
    dt = f.dtype.type
    g = synth.rng(seed).normal(size=f.shape).astype(dt)
    gf = A.eikonal_grad(dev(g), dev(u), dev(f), sx, sy, h).cpu().numpy()
    ns = A.ops.last_info["n_singular"]
    gr, _, nr = oracle.eikonal2d_grad(g, u, f, sx, sy, h, dtype=dt)
    assert ns == nr
    tol = 4000 * np.finfo(dt).eps
    assert np.abs(gf - gr).max() <= tol * np.abs(gr).max()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [
    (2, 2), (2, 9), (3, 64), (63, 65), (64, 64), (65, 64), (65, 65), (66, 130), (129, 70),
    (101, 122), (135, 136), (300, 37), (513, 520), (530, 512), (341, 330), (1030, 40)])
def test_2d_bit_exact(shape, dt):
    f = 1.0 / synth.gaussians_2d(shape, 1.0, seed=sum(shape))
    r = synth.rng(sum(shape))
    check(f, int(r.integers(1, shape[1] + 1)), int(r.integers(1, shape[0] + 1)), 0.7, dt)
    check(f, shape[1], 1, 0.7, dt)


def test_2d_more_rows_than_bands():
    f = 1.0 / synth.gaussians_2d((1030, 1026), 1.0, seed=3)
    check(f, 500, 17, 1.0, np.float64)


@pytest.mark.parametrize("value", [np.nan, 0.0, 1e-300, 1e90, -0.5])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_2d_any_slowness(value, dt):
    f = np.ones((70, 33))
    f[40:43, 5:9] = value
    with np.errstate(over="ignore"):
        f = f.astype(dt)
    import adtomo_hip as A
    ref, it, _, _ = oracle.eikonal2d(f, 3, 60, 1.0, dtype=dt)
    u = A.eikonal(dev(f), 3, 60, 1.0).cpu().numpy()
    assert np.array_equal(u, ref, equal_nan=True) and A.ops.last_info["iterations"] == it


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(90, 110), (150, 140), (340, 325), (400, 300)])
def test_2d_adjoint_of_any_field(shape, dt):
    """Random values: a third of the nodes resolve in the first level (more than
    the LDS queue holds), many are singular."""
    r = synth.rng(shape[0])
    u = r.uniform(1.0, 2.0, size=shape).astype(dt)
    check_adjoint(u, r.uniform(0.5, 1.5, size=shape).astype(dt), 7, 80, 1.0)
