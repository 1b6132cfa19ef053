"""Materials set while coefficient compression is off, which is turned on again: the
next solve reads theirs, not the index of those before."""
import numpy as np
import pytest

from tests.cases import build_sim, strip_case
from tests.test_gpu_resident import _solve

pytestmark = pytest.mark.gpu


def _sim(case):
    sim = build_sim(case)
    sim._lib.emf_set_resident(sim._h, 0, 0)
    sim.fixed_n0 = 60
    return sim


def test_materials_set_without_compression():
    first, second = strip_case(40, 32, 24, w=5), strip_case(40, 32, 24, w=5, core=(0.3, 0.3))
    ref, _ = _solve(_sim(second), second)
    sim = _sim(first)
    before, _ = _solve(sim, first)
    sim._lib.emf_set_compression(sim._h, 0)
    sim.set_material_arrays(second["mats"][:3], second["mats"][3:])
    sim._lib.emf_set_compression(sim._h, 1)
    got, _ = _solve(sim, second)
    assert not np.array_equal(before[2], ref[2])
    assert all(np.array_equal(x, y) for x, y in zip(got, ref))
