"""Solves after a stalled resident launch (polls limited to one): reported, left
to the passes for one solve, then two, and tried again."""
import ctypes
import warnings

import numpy as np
import pytest

from tests.cases import all_fields, build_sim, rel_l2, strip_case
from tests.test_gpu_resident import TOL, _boxes, _solve

pytestmark = pytest.mark.gpu


def _warned(sim, case):
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        sim._register(sim._sources)
        sim._solve(0)
    return all_fields(sim, case), any(w.category is RuntimeWarning and "resident" in str(w.message)
                                      for w in seen)


def test_resident_steps_are_tried_again_after_a_stall():
    case = strip_case(40, 32, 24, w=5)
    sim = build_sim(case)
    sim.fixed_n0 = 100
    sim._lib.emf_set_resident(sim._h, 0, 0)
    ref, _ = _solve(sim, case)
    sim._lib.emf_set_resident(sim._h, 1, 1)
    n = ctypes.c_int()
    for stalls, expect in enumerate((True, False, True, False, False, True)):
        assert (_boxes(sim) > 1) == expect, stalls
        got, warned = _warned(sim, case)
        assert warned == expect
        assert all(np.array_equal(x, y) for x, y in zip(got, ref))
    sim._lib.emf_resident_stalls(sim._h, ctypes.byref(n))
    assert n.value == 3 and _boxes(sim) == 0
    sim._lib.emf_set_resident(sim._h, 1, 0)
    assert _boxes(sim) > 1
    got, warned = _warned(sim, case)
    assert not warned and _boxes(sim) > 1
    assert max(rel_l2(x, y) for x, y in zip(got, ref)) <= TOL
