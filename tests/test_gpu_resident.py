"""Resident solves (k_resident: the state on chip, faces exchanged between
work-groups) against the two passes: the same solve, fields to roundoff."""
import ctypes
import warnings

import numpy as np
import pytest

from tests.cases import all_fields, build_sim, random_case, rel_l2, strip_case

pytestmark = pytest.mark.gpu

# both paths carry the rounding of ~200 steps (each within 1e-14 of the oracle)
TOL = 1e-12


def _solve(sim, case):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        sim._register(sim._sources)
        sim._solve(0)
    return all_fields(sim, case), dict(sim.last_solve)


def _boxes(sim):
    n = ctypes.c_int()
    sim._lib.emf_resident(sim._h, ctypes.byref(n))
    return n.value


# one box, single planes, spare planes (Nz not a multiple), every plane count,
# odd sizes, boxes at and inside the slabs, and the largest grids of each form
@pytest.mark.parametrize("dims,w,kw", [
    ((3, 2, 2), (0,) * 6, {}),
    ((9, 7, 5), (2, 2, 2, 2, 1, 1), {}),
    ((24, 20, 16), (4,) * 6, dict(bc="0H0")),
    ((70, 37, 23), (5, 4, 3, 6, 4, 5), dict(bc="EH0", nsrc=3)),
    ((67, 65, 61), (8, 7, 9, 8, 7, 9), dict(bc="HEH", nsrc=70)),
    ((131, 50, 47), (6, 6, 0, 6, 6, 6), dict(bc="0E0")),
    ((127, 79, 59), (10,) * 6, {}),
    ((33, 29, 31), (4,) * 6, dict(ceps=True)),
    ((61, 53, 47), (5, 4, 3, 6, 4, 5), dict(ceps=True, mu=True, bc="E0H")),
    ((97, 41, 53), (6,) * 6, dict(mu=True)),
])
def test_resident_solve_equals_two_passes(dims, w, kw):
    kw = dict(kw)
    mu = kw.pop("mu", False)
    case = random_case(*dims, w=w, seed=sum(dims), mu_rand=mu, **kw)
    sim = build_sim(case)
    sim.fixed_n0 = 71                 # a full launch and a partial one
    assert _boxes(sim) > 0
    got, a = _solve(sim, case)
    sim._lib.emf_set_resident(sim._h, 0, 0)
    assert _boxes(sim) == 0
    ref, b = _solve(sim, case)
    errs = [rel_l2(x, y) for x, y in zip(got, ref)]
    print(dims, ["%.1e" % e for e in errs])
    assert a["steps"] == b["steps"] and max(errs) <= TOL, errs


def test_converged_solves_and_changes_between_them():
    """Converged solves stop at the same step with the same checks, also after
    the boxes of the split change (CPML widths, sources) and on a second solve."""
    case = strip_case(40, 32, 24, w=5)
    sim = build_sim(case)
    for widths in ([5] * 6, [3, 4, 5, 6, 4, 3]):
        sim.w_pml = [(v + 1e-9) * case["d"] for v in widths]
        sim._lib.emf_set_resident(sim._h, 1, 0)
        runs = [_solve(sim, case) for _ in range(2)]
        sim._lib.emf_set_resident(sim._h, 0, 0)
        ref, info = _solve(sim, case)
        for got, a in runs:
            assert a["n0"] == info["n0"] and a["nchecks"] == info["nchecks"]
            errs = [rel_l2(x, y) for x, y in zip(got, ref)]
            assert max(errs) <= TOL, errs
        assert all(np.array_equal(x, y) for x, y in zip(runs[0][0], runs[1][0]))


def test_stalled_launch_is_repeated_with_the_passes():
    """A launch whose polls give up (a limit of one poll) leaves the solve to
    the two passes, from the start; later solves of the handle use them too."""
    case = strip_case(40, 32, 24, w=5)
    sim = build_sim(case)
    sim.fixed_n0 = 100
    sim._lib.emf_set_resident(sim._h, 0, 0)
    ref, _ = _solve(sim, case)
    sim._lib.emf_set_resident(sim._h, 1, 1)
    assert _boxes(sim) > 1
    got, _ = _solve(sim, case)
    assert _boxes(sim) == 0
    assert all(np.array_equal(x, y) for x, y in zip(got, ref))
    sim._lib.emf_set_resident(sim._h, 1, 0)
    got, _ = _solve(sim, case)
    assert _boxes(sim) > 1
    assert max(rel_l2(x, y) for x, y in zip(got, ref)) <= TOL

