"""The objective's kernels at the edges of their work splits: arrays that start
off a 16-byte boundary or end within a piece, more stations and arrays than one
table holds, smoothing runs cut by the grid's end and windows as wide as the
grid, receivers in more workgroups than one.  Fills, times, sums and misfit
gradients bit for bit; smoothing within 1e-13 (box sums of up to 125 terms)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import objective as OO  # noqa: E402


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def at_offset(shape, k):
    import torch
    n = int(np.prod(shape))
    return torch.full((n + 8,), -7.0, dtype=torch.float64, device="cuda")[k:k + n].view(shape)


@pytest.mark.parametrize("shape,count", [((2, 2, 2), 1), ((17, 13, 9), 70), ((40, 50, 30), 3)])
def test_source_times(shape, count):
    from adtomo_hip import objective as O
    r = np.random.default_rng(count)
    vel0 = r.uniform(3, 8, shape)
    st = [tuple(float(r.uniform(1, s)) for s in shape) for _ in range(count)]
    st[0] = tuple(float(s) for s in shape)
    out = [at_offset(shape, e % 3) for e in range(count)]
    O.source_u0(st, dev(vel0), 0.5, 1.3, out=out)
    for s, u in zip(st, out):
        np.testing.assert_array_equal(u.cpu().numpy(), OO.source_u0(shape, *s, vel0, 0.5, 1.3))
        tail = u.storage_offset() + u.numel()
        assert float(u.as_strided((1,), (1,), tail)[0]) == -7.0


@pytest.mark.parametrize("shape,ns,ne", [((9, 8, 7), 2, 2100), ((30, 41, 23), 70, 60)])
def test_misfit_parts(shape, ns, ne):
    from adtomo_hip import objective as O
    r = np.random.default_rng(ne)
    us = [r.uniform(0, 10, shape) for _ in range(ns)]
    rx, ry, rz = (r.uniform(1, s, ne) for s in shape)
    tobs, w = r.uniform(0, 10, (ns, ne)), r.uniform(0.2, 2.0, (ns, ne))
    tobs[:, ::7] = -1.0
    out = O.misfit([dev(u) for u in us], rx, ry, rz, [dev(t) for t in tobs], [dev(x) for x in w],
                   grad_out=[at_offset(shape, e % 3) for e in range(ns)])
    for s in range(ns):
        tcal, L, g = OO.misfit(us[s], rx, ry, rz, tobs[s], w[s])
        np.testing.assert_array_equal(out["tcal"][s].cpu().numpy(), tcal)
        np.testing.assert_array_equal(out["grad_u"][s].cpu().numpy(), g)
        assert abs(float(out["loss"][s]) - L) <= 1e-13 * abs(L)


@pytest.mark.parametrize("shape,sh,sv", [
    ((3, 3, 3), 3, 3), ((8, 5, 4), 3, 3), ((9, 4, 3), 3, 3), ((65, 33, 20), 3, 3), ((5, 5, 5), 5, 5),
    ((65, 33, 20), 5, 3)])
def test_smoothing_runs(shape, sh, sv):
    from adtomo_hip import objective as O
    r = np.random.default_rng(sum(shape))
    fvar = r.uniform(3, 8, shape)
    val, g = O.smooth_l1(dev(fvar), sh, sv, 0.3)
    rval, rg = OO.smooth_l1(fvar, sh, sv, 0.3)
    assert abs(float(val) - rval) <= 1e-13 * abs(rval) + 1e-13
    assert np.abs(g.cpu().numpy() - rg).max() <= 1e-13


@pytest.mark.parametrize("count", [1, 256, 257])
def test_sum_of_many_arrays(count):
    from adtomo_hip import objective as O
    r = np.random.default_rng(count)
    arrs = [r.normal(size=(3, 7, 5)) for _ in range(count)]
    ref = arrs[0].copy()
    for a in arrs[1:]:
        ref = ref + a
    np.testing.assert_array_equal(O.sum_arrays([dev(a) for a in arrs]).cpu().numpy(), ref)
