"""A batched call takes each event's box from its slowness; an array beside it that is
smaller (in bytes) is refused on the host, before any kernel could run past its end.
On the CPU: tensors that say they are on the device, none of which is ever read."""
import pytest
import torch

import adtomo_hip as A
from adtomo_hip import ops


class OnDevice(torch.Tensor):
    is_cuda = True


def arr(*shape, dtype=torch.float64):
    return torch.zeros(shape, dtype=dtype).as_subclass(OnDevice)


BOX = (6, 5, 4)


def table(**arrays):
    f = arr(*BOX)
    a = dict(u0=arr(*BOX), us=arr(*BOX), grad_us=arr(*BOX), grad_u0s=arr(*BOX), grad_fs=arr(*BOX))
    a.update(arrays)
    two = {k: [arr(*BOX), x] for k, x in a.items()}  # the second event's
    return ops._event_table(two["u0"], [arr(*BOX), f], [0.5] * 2, [1e-3] * 2, two["grad_us"],
                            two["us"], two["grad_u0s"], two["grad_fs"])


def test_arrays_of_the_box_are_taken():
    tab, dtype = table()
    assert dtype == torch.float64 and (tab[1].m, tab[1].n, tab[1].l) == BOX
    table(u0=arr(120), us=arr(200), grad_us=arr(7, 5, 4))  # as long as they reach


@pytest.mark.parametrize("which", ["u0", "us", "grad_us", "grad_u0s", "grad_fs"])
@pytest.mark.parametrize("small", [arr(6, 5, 3), arr(*BOX, dtype=torch.float32), arr(0)])
def test_a_smaller_array_is_refused(which, small):
    with pytest.raises(ValueError, match="event 1"):
        table(**{which: small})


def test_the_entry_points_refuse_it():
    u0s, fs = [arr(*BOX), arr(5, 5, 4)], [arr(*BOX)] * 2
    with pytest.raises(ValueError, match="event 1: u0"):
        A.eikonal3d_batched(u0s, fs, [0.5] * 2, [1e-3] * 2)
    with pytest.raises(ValueError, match="event 1: u0"):
        A.EikonalGraph(u0s, fs, [0.5] * 2, [1e-3] * 2)
    with pytest.raises(ValueError, match="event 1: u0"):
        ops.selftest_forward(u0s, fs, [0.5] * 2, [1e-3] * 2)
