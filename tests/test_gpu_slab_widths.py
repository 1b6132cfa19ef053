"""Deep resident boxes and slabs of different widths on the two faces of an axis.
The grid fills the chip (256 boxes of 512 columns of 10 planes), so there are only
two ways to split it, into one box or two along its short axis."""
import numpy as np
import pytest

from tests.cases import build_sim, random_case, rel_l2
from tests.test_gpu_resident import TOL, _boxes, _solve

pytestmark = pytest.mark.gpu


def _case(axis, widths):
    dims = (32, 256, 160) if axis == 0 else (256, 32, 160)
    w = [8] * 6
    w[2 * axis:2 * axis + 2] = widths
    return random_case(*dims, w=w, seed=5 + axis, mu_rand=False)


@pytest.mark.parametrize("axis", [0, 1])
def test_boxes_that_meet_slabs_of_two_widths_are_refused(axis):
    """17 and 9 of 32 cells: in either split some box meets both slabs."""
    case = _case(axis, (17, 9))
    sim = build_sim(case)
    assert _boxes(sim) == 0
    sim.fixed_n0 = 5
    got, _ = _solve(sim, case)
    sim._lib.emf_set_resident(sim._h, 0, 0)
    ref, _ = _solve(sim, case)
    assert all(np.array_equal(x, y) for x, y in zip(got, ref))


@pytest.mark.parametrize("axis,widths", [(0, (16, 9)), (1, (16, 9)), (0, (9, 9)), (1, (15, 15)), (0, (17, 0))])
def test_boxes_that_meet_one_width_are_taken(axis, widths):
    case = _case(axis, widths)
    sim = build_sim(case)
    assert _boxes(sim) == 256
    sim.fixed_n0 = 71
    got, _ = _solve(sim, case)
    sim._lib.emf_set_resident(sim._h, 0, 0)
    ref, _ = _solve(sim, case)
    errs = [rel_l2(x, y) for x, y in zip(got, ref)]
    assert max(errs) <= TOL, errs
