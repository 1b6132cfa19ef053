"""Resident solves of grids whose psi and coefficients stay in memory (deep
boxes) against the two passes: the fields of a solve, and of steps taken after
it, which start from the psi that the solve left."""
import ctypes

import numpy as np
import pytest

from tests.cases import build_sim, random_case, rel_l2
from tests.test_gpu_resident import TOL, _boxes, _solve

pytestmark = pytest.mark.gpu


# just past what registers hold with psi (655 thousand cells, 393 thousand with
# complex eps), spare planes, slabs of different widths, boxes that meet both
# faces of an axis, no slabs on an axis, every plane count, the largest grids
@pytest.mark.parametrize("dims,w,kw", [
    ((118, 78, 72), (10,) * 6, {}),
    ((127, 91, 61), (5, 9, 7, 6, 8, 4), dict(bc="0H0")),
    ((180, 60, 80), (10,) * 6, dict(bc="E0H", nsrc=5)),
    ((44, 150, 131), (9, 9, 0, 0, 6, 7), {}),
    ((151, 97, 71), (8, 7, 9, 8, 0, 9), {}),
    ((128, 96, 90), (10,) * 6, {}),
    ((120, 72, 55), (6, 5, 4, 6, 7, 5), dict(ceps=True, bc="H0E")),
    ((173, 101, 67), (10,) * 6, dict(ceps=True)),
])
def test_deep_solve_equals_two_passes(dims, w, kw):
    case = random_case(*dims, w=w, seed=sum(dims), mu_rand=False, **kw)
    cells = np.prod(dims)
    assert cells > (393216 if case["ceps"] else 655360)
    sim = build_sim(case)
    sim.fixed_n0 = 71
    assert _boxes(sim) > 0
    out = np.zeros(3)

    def more(info):
        sim._lib.emf_time_steps(sim._h, info["steps"], 9, 0, 0, out.ctypes.data_as(ctypes.c_void_p))
        return sim.time_fields()
    got, a = _solve(sim, case)
    got += list(more(a))
    sim._lib.emf_set_resident(sim._h, 0, 0)
    ref, b = _solve(sim, case)
    ref += list(more(b))
    errs = [rel_l2(x, y) for x, y in zip(got, ref)]
    print(dims, ["%.1e" % e for e in errs])
    assert a["steps"] == b["steps"] and max(errs) <= TOL, errs


def test_two_slab_widths_in_one_box_take_the_passes():
    """A box that meets both faces of an axis with slabs of different widths has
    no deep kernel: 60 rows of x in one box."""
    case = random_case(18, 160, 240, w=(9, 8, 8, 8, 8, 8), seed=1, mu_rand=False)
    sim = build_sim(case)
    same = random_case(18, 160, 240, w=(8,) * 6, seed=1, mu_rand=False)
    boxes = _boxes(sim)
    sim2 = build_sim(same)
    if boxes == 0:
        assert _boxes(sim2) > 0
    sim.fixed_n0 = sim2.fixed_n0 = 71
    got, _ = _solve(sim, case)
    sim._lib.emf_set_resident(sim._h, 0, 0)
    ref, _ = _solve(sim, case)
    assert max(rel_l2(x, y) for x, y in zip(got, ref)) <= TOL
