"""The grouping of steps into launches that pf_advance_* makes
(pf_launch_steps), on the CPU."""
import ctypes

import pytest

from pfpa import lib
from pfpa import model as M
from pfpa.sim import iter_launches, plan_launches, segments

FIVE = M.five_point_mask(0.25e-9, 0.25e-9)
NINE = M.nine_point_mask(0.25e-9, 0.325e-9)
LOPSIDED = [0.0, 1.0, 0.0, 1.2, -4.0, 0.8, 0.0, 1.0, 0.0]


def _k(nx, ny, mask, steps, most):
    return lib().pf_launch_steps(nx, ny, (ctypes.c_double * 9)(*mask), steps, most)


@pytest.mark.parametrize("most", [1, 2, 3, 4])
def test_steps_of_a_launch(most):
    for steps in (0, 1, 2, 3, 4, 5, 1 << 40):
        want = min(steps, most)
        assert _k(100, 80, FIVE, steps, most) == want
        assert _k(100, 80, NINE, steps, most) == (2 if want == 3 else want)   # no three-step kernel
        assert _k(100, 80, LOPSIDED, steps, most) == min(steps, 1)
        # interiors below 4x4 take three steps at most, below 3x3 one
        for nx, ny in ((5, 80), (100, 5)):
            assert _k(nx, ny, FIVE, steps, most) == min(want, 3)
        for nx, ny in ((4, 80), (100, 4)):
            assert _k(nx, ny, FIVE, steps, most) == min(steps, 1)


def test_refused():
    assert lib().pf_launch_steps(100, 80, None, 4, 4) == 0
    for most in (-1, 0, 5):
        assert _k(100, 80, FIVE, 4, most) == 0
        with pytest.raises(ValueError):
            plan_launches(0, 4, most)


def test_plans_of_other_masks():
    def plan(mask, n, most=4):
        return [k for k, _ in iter_launches(0, n, most, 0, 100, 80, mask)]

    assert plan(NINE, 11) == [4, 4, 2, 1] and plan(NINE, 7, 3) == [2, 2, 2, 1]
    assert plan(LOPSIDED, 3) == [1, 1, 1]
    assert list(iter_launches(0, 8, 4, 5, 100, 80, NINE)) == [(1, True), (4, False), (1, True),
                                                              (2, False)]


def test_segments():
    assert list(segments(0, 0, 5)) == [] and list(segments(3, 4)) == [(4, False)]
    assert list(segments(0, 12, 5)) == [(1, True), (4, False), (1, True), (4, False), (1, True),
                                        (1, False)]
    assert list(segments(7, 2, 5)) == [(2, False)]
    assert list(segments(2, 3, 1)) == [(1, True)] * 3


def test_a_mask_may_be_an_array():
    import numpy as np
    assert [k for k, _ in iter_launches(0, 5, 4, 0, 100, 80, np.array(NINE))] == [4, 1]
