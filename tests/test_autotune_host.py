"""What tune_solver applies where solves run resident, and from its cache before
the materials are set (CPU only, with a stand-in library)."""
import ctypes
import types

import pytest

from emopt_amd import autotune


class Lib:
    """Two passes, but `fused` is the fastest step kernel; resident in kind 1."""

    def __init__(self, fits):
        self.fits = fits
        self.kind = (1, 4, 2, 3)

    def emf_set_tuning(self, h, *t):
        self.kind = tuple(t)

    def emf_resident(self, h, boxes):
        ctypes.cast(boxes, ctypes.POINTER(ctypes.c_int))[0] = 8 if self.fits and self.kind[0] == 1 else 0

    def emf_reset_pml(self, h):
        pass

    emf_zero_fields = emf_reset_pml

    def emf_time_steps(self, h, n, steps, tn, conv, out):
        ms = {(2, 8, 4, 0): 0.5, (1, 2, 4, 3): 0.8}.get(self.kind, 1.0)
        ctypes.cast(out, ctypes.POINTER(ctypes.c_double))[0] = ms * steps


def _sim(fits, ready):
    def build():
        assert ready, "built before the materials were set"
    return types.SimpleNamespace(Nx=7, Ny=6, Nz=5, Tn=4, _complex_eps=0, _h=1, _lib=Lib(fits),
                                 _mats_ready=ready, build=build, _sources=[],
                                 _register=lambda s: None)


@pytest.mark.parametrize("fits,used", [(True, (1, 2, 4, 3)), (False, (2, 8, 4, 0))])
def test_fastest_kernel_that_keeps_resident_solves(fits, used, monkeypatch):
    monkeypatch.setattr(autotune, "_cache", {})
    sim = _sim(fits, True)
    best, times = autotune.tune_solver(sim)
    assert best == (2, 8, 4, 0) and len(times) == len(autotune.SOLVE_CANDIDATES)
    assert sim._lib.kind == used


@pytest.mark.parametrize("best,fits,used", [
    ((2, 8, 4, 0), True, (1, 4, 2, 3)), ((2, 8, 4, 0), False, (2, 8, 4, 0)),
    ((1, 2, 4, 3), True, (1, 2, 4, 3))])
def test_cached_choice_before_the_materials(best, fits, used, monkeypatch):
    sim = _sim(fits, False)
    monkeypatch.setattr(autotune, "_cache", {autotune._key(sim): list(best)})
    assert autotune.tune_solver(sim) == (best, {})
    assert sim._lib.kind == used
