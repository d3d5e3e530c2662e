"""The 2D forward on grids so long that a wave waits for most of a sweep of the wave
before it: the waits of fwd2_band_kernel are bounded by the time without any
progress, not by the time of a sweep.  Bit for bit against the CPU oracle, the long
axis along x and along y, with 2 and with 65 rows (one and two bands)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle  # noqa: E402


@pytest.mark.parametrize("shape, dt", [
    ((2, 1500000), np.float64), ((1500000, 2), np.float32), ((65, 400001), np.float32)])
def test_2d_long_grid(shape, dt):
    import torch
    import adtomo_hip as A
    # slowness that varies over some 10^5 nodes: a few iterations
    f = 1.0 + 0.3 * np.sin(np.arange(max(shape)) * 1e-5)
    f = np.repeat(f[:, None], min(shape), axis=1)
    f = np.ascontiguousarray(f if shape[0] > shape[1] else f.T).astype(dt)
    sx = max(1, shape[1] // 3)
    ref, it, err, _ = oracle.eikonal2d(f, sx, 1, 0.01, dtype=dt)
    u = A.eikonal(torch.from_numpy(f).to("cuda"), sx, 1, 0.01).cpu().numpy()
    assert A.ops.last_info["iterations"] == it and A.ops.last_info["fault"] == 0
    w = np.uint64 if dt == np.float64 else np.uint32
    assert np.array_equal(u.view(w), ref.view(w))
