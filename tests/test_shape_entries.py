"""boundary_deps on structured materials whose entries are not one per primitive
(CPU only): an object added twice, polygons with nothing left of them, and on
solvers that cannot take the call.  The lists that go to the device are checked
with a stand-in library."""
import ctypes
import types

import numpy as np
import pytest

from emopt_amd import _lib, grid
from emopt_amd.shape import boundary_deps, rect_edge_velocity

SHIFTS = ((0.5, 0.0, -0.5), (0.0, 0.5, -0.5), (0.0, 0.0, 0.0))
N, D = (20, 16, 12), 0.1


class Lists:
    """emf_shape_deps: keeps the lists it is given, then has the host compute."""

    def emf_shape_deps(self, h, recs, nrings, vx, vy, nv, dx, dy, br, bi, off, lst, mine, nseg,
                       edges, nedges, box, shifts, out, limit):
        def ints(p, n):
            return list((ctypes.c_int * n).from_address(p))
        self.off = ints(off, nseg + 1)
        self.rings = [ints(lst, self.off[-1])[a:b] for a, b in zip(self.off, self.off[1:])]
        self.mine = ints(mine, nseg)
        ctypes.cast(limit, ctypes.POINTER(ctypes.c_int))[0] = 1


def _sims():
    host = types.SimpleNamespace(Nx=N[0], Ny=N[1], Nz=N[2], YEE_SHIFTS=SHIFTS)
    dev = types.SimpleNamespace(**vars(host), _h=1, _lib=Lists())
    return host, dev


def _twice():
    """A moving rectangle added over (0, 1.2) and (0.4, 0.8), and one of the same
    layer between them: three segments, the middle one with the object twice."""
    eps = grid.StructuredMaterial3D(N[0] * D, N[1] * D, N[2] * D, D, D, D, background=1.0)
    p = grid.Rectangle(1.0, 0.8, 0.73, 0.55, material_value=9.0, layer=1)
    q = grid.Rectangle(1.3, 0.8, 0.57, 0.35, material_value=4.0, layer=1)
    eps.add_primitive(p, 0.0, 1.2)
    eps.add_primitive(q, 0.0, 1.2)
    eps.add_primitive(p, 0.4, 0.8)
    return eps, p


def test_moving_object_added_twice_has_one_place_per_segment():
    eps, p = _twice()
    _, dev = _sims()
    boundary_deps(dev, eps, p, rect_edge_velocity("xr"))
    assert dev._lib.mine == [0, 2, 0]        # the last of its entries in the segment
    assert len(dev._lib.rings) == 3
    first = dev._lib.rings[0][0]
    assert [r[m] for r, m in zip(dev._lib.rings, dev._lib.mine)][::2] == [first, first]


def _dense(deps):
    out = np.zeros((3, N[0] * N[1] * N[2]), dtype=complex)
    np.add.at(out, deps[:2], deps[2])
    return out


def test_moving_object_added_twice_host_rule():
    """The segments are independent, and in the middle one its last entry moves,
    with the first where it is: the sum of three materials, a copy for the first."""
    eps, p = _twice()
    host, _ = _sims()
    got = _dense(boundary_deps(host, eps, p, rect_edge_velocity("xr")))
    want = np.zeros_like(got)
    for z1, z2, copy in ((0.0, 0.4, False), (0.4, 0.8, True), (0.8, 1.2, False)):
        part = grid.StructuredMaterial3D(N[0] * D, N[1] * D, N[2] * D, D, D, D, background=1.0)
        if copy:
            part.add_primitive(grid.Rectangle(1.0, 0.8, 0.73, 0.55, material_value=9.0, layer=1), z1, z2)
        part.add_primitive(grid.Rectangle(1.3, 0.8, 0.57, 0.35, material_value=4.0, layer=1), z1, z2)
        mine = grid.Rectangle(1.0, 0.8, 0.73, 0.55, material_value=9.0, layer=1 if copy else 0)
        part.add_primitive(mine, z1, z2)
        want += _dense(boundary_deps(host, part, mine, rect_edge_velocity("xr")))
    assert np.abs(want).max() > 0
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-12 * np.abs(want).max())


@pytest.mark.parametrize("device", [False, True])
def test_polygons_with_nothing_left_do_not_count(device):
    """A polygon of fewer than three vertices is no ring: the derivative is that
    without it, whichever of them comes first."""
    host, dev = _sims()
    res = []
    for empty in (False, True):
        eps = grid.StructuredMaterial3D(N[0] * D, N[1] * D, N[2] * D, D, D, D)
        p = grid.Rectangle(1.0, 0.8, 0.73, 0.55, material_value=9.0, layer=2)
        if empty:
            for layer in (1, 3):
                g = grid.Polygon([0.2, 0.9, 0.5], [0.2, 0.3, 0.9], material_value=4.0, layer=layer)
                g.xs, g.ys = g.xs[:2], g.ys[:2]
                eps.add_primitive(g, 0.0, 1.2)
        eps.add_primitive(p, 0.0, 1.2)
        res.append(boundary_deps(dev if device else host, eps, p, rect_edge_velocity("xr")))
        if device:
            assert dev._lib.mine == [0]
    for a, b in zip(*res):
        assert len(a) > 0 and np.array_equal(a, b)


@pytest.mark.parametrize("code", [_lib.ERR_STATE, _lib.ERR_NOMEM, _lib.ERR_HIP])
def test_refused_by_the_solver(code):
    """A solver that is a batch member or busy, or a device without room, leaves
    the derivative to the host; other errors are raised."""
    eps, p = _twice()
    host, dev = _sims()

    def refuse(*args):
        raise _lib.EmfError("refused", code)
    dev._lib.emf_shape_deps = refuse
    if code == _lib.ERR_HIP:
        with pytest.raises(_lib.EmfError):
            boundary_deps(dev, eps, p, rect_edge_velocity("xr"))
        return
    for a, b in zip(boundary_deps(dev, eps, p, rect_edge_velocity("xr")),
                    boundary_deps(host, eps, p, rect_edge_velocity("xr"))):
        assert np.array_equal(a, b)
