"""A cached tuning applied to a solver whose materials are not set yet, on the GPU."""
import ctypes
import warnings

import pytest

from emopt_amd import autotune
from emopt_amd.fdtd import FDTD
from tests.cases import span

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,fits", [((24, 20, 16), True), ((200, 130, 100), False)])
def test_cached_choice_needs_no_materials(N, fits, monkeypatch):
    d = 0.05
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        sim = FDTD(*(span(n, d) for n in N), d, d, d, 1.55)
    sim.w_pml = [2.5 * d] * 6
    boxes = ctypes.c_int()
    sim._lib.emf_resident(sim._h, ctypes.byref(boxes))
    assert (boxes.value > 0) == fits
    monkeypatch.setattr(autotune, "_cache", {autotune._key(sim): [2, 8, 4, 0]})
    assert autotune.tune_solver(sim) == ((2, 8, 4, 0), {})
    sim._lib.emf_resident(sim._h, ctypes.byref(boxes))
    assert (boxes.value > 0) == fits
    sim._lib.emf_set_wide_offsets(sim._h, 1)
    sim._lib.emf_resident(sim._h, ctypes.byref(boxes))
    assert boxes.value == 0
