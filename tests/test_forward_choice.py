"""The forward kernel that the library chooses for a batch (no device is needed):
on either side of the number of events from which one workgroup each is the faster
one, and where the others stay faster by far (times of all forms beside
choose_forward in csrc/abi.hip)."""
import pytest

from adtomo_hip import ops

MODES = [("float64", False), ("float32", False), ("float32", True)]


def forms(shapes, mode):
    return set(ops.selftest_forward_forms(shapes, mode[0], compute_f64=mode[1]))


@pytest.mark.parametrize("mode", MODES, ids=["f64", "f32", "mixed"])
def test_equal_full_boxes(mode):
    box = (128, 128, 64)
    for n in (64, 128, 160):
        assert forms([box] * n, mode) == {"wide"}, n
    for n in (176, 192, 208, 224, 240, 256):
        assert forms([box] * n, mode) == {"one"}, n


def test_equal_boxes_of_one_band():
    for box in [(60, 128, 64), (64, 128, 60)]:
        assert forms([box] * 64, MODES[0]) == {"wide"}
        assert forms([box] * 250, MODES[0]) == {"one"}


def test_equal_boxes_of_odd_columns():
    f64, mixed = MODES[0], MODES[2]
    for box, n in [((93, 95, 59), 206), ((90, 120, 57), 200), ((126, 126, 64), 200)]:
        assert forms([box] * n, f64) == {"one"}, (box, n)
    for box, n in [((48, 33, 57), 247), ((40, 60, 63), 256), ((33, 160, 60), 256),
                   ((76, 110, 61), 171), ((64, 64, 61), 200), ((50, 50, 64), 256)]:
        assert forms([box] * n, f64) == {"wide"}, (box, n)
    assert forms([(14, 160, 9)] * 338, mixed) == {"team"}
    assert forms([(86, 93, 62)] * 213, mixed) == {"wide"}
    assert forms([(24, 20, 12)] * 400, f64) == {"team"}


@pytest.mark.parametrize("mode", MODES, ids=["f64", "f32", "mixed"])
def test_boxes_that_stay_on_several_workgroups(mode):
    for box, n in [((200, 200, 80), 200), ((101, 90, 47), 256), ((96, 100, 48), 224),
                   ((100, 100, 100), 256), ((64, 64, 64), 256), ((128, 128, 96), 250)]:
        assert forms([box] * n, mode) == {"wide"}, (box, n)
    uneven = [(48 + 5 * e % 81, 48 + 7 * e % 81, 24 + 3 * e % 41) for e in range(256)]
    assert forms(uneven, mode) == {"wide"}
