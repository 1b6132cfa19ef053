"""FDTD.grad_assemble checks that every entry array covers the parameter indices
before their pointers go to the library (CPU only, with a stand-in library)."""
import ctypes
import types

import numpy as np
import pytest

from emopt_amd.fdtd import FDTD


class Reader:
    """The two entry points: read n entries of each array, as the library does."""

    def __init__(self):
        self.entries = []

    def emf_grad_assemble(self, h, n, pidx, comp, cell, deps, nparam, step, grad):
        def get(p, typ, m):
            return np.array((typ * m).from_address(p.value))
        self.entries.append((get(pidx, ctypes.c_int32, n), get(comp, ctypes.c_int32, n),
                             get(cell, ctypes.c_int64, n), get(deps, ctypes.c_double, 2 * n)))

    emf_grad_assemble_noalloc = emf_grad_assemble


def _sim():
    return types.SimpleNamespace(_lib=Reader(), _h=1)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("pidx", [[0, 0, 1, 2], [2, 0, 1, 0]])
@pytest.mark.parametrize("short", ["comp", "cell", "deps"])
def test_short_arrays_are_refused(short, pidx, noalloc):
    a = dict(comp=[0, 1, 2, 0], cell=[5, 6, 7, 8], deps=[1j, 2, 3, 4])
    a[short] = a[short][:2]
    sim = _sim()
    with pytest.raises(IndexError):
        FDTD.grad_assemble(sim, pidx, a["comp"], a["cell"], a["deps"], 3, noalloc=noalloc)
    assert sim._lib.entries == []


@pytest.mark.parametrize("pidx", [[0, 0, 1, 2], [2, 0, 1, 0]])
def test_entries_reach_the_library_grouped(pidx):
    """Entries beyond those of pidx are left out, columns are taken as lists."""
    sim = _sim()
    comp, cell, deps = np.arange(5) % 3, np.arange(5) + 10, (np.arange(5) + 1j)[:, None]
    FDTD.grad_assemble(sim, pidx, comp, cell, deps, 3)
    order = np.argsort(pidx, kind="stable")
    p, c, g, d = sim._lib.entries[0]
    assert np.array_equal(p, np.array(pidx)[order]) and np.array_equal(c, comp[order])
    assert np.array_equal(g, cell[order]) and np.array_equal(d.view(complex), deps[order, 0])


def test_parameter_indices_are_a_list():
    with pytest.raises(ValueError):
        FDTD.grad_assemble(_sim(), [[0, 1]], [0, 0], [1, 2], [1, 1], 2)
