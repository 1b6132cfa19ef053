"""Analytic shape derivatives on the GPU (emf_shape_deps) against the host rule
they repeat operation for operation: the same entries, in the same order, with
the same doubles -- rectangles and polygons, edges on and off cell boundaries,
overlaps before and after in priority, several z segments, moving parts outside
the grid -- and the host's answer where a cell counts more primitives than the
device holds."""
import types
import warnings

import numpy as np
import pytest

from emopt_amd.fdtd import FDTD
from emopt_amd.grid import ConstantMaterial3D, Ellipse, Polygon, Rectangle, StructuredMaterial3D
from emopt_amd.shape import boundary_deps, polygon_vertex_velocity, rect_edge_velocity
from tests.cases import span

pytestmark = pytest.mark.gpu
D, N = 0.05, (20, 17, 8)


def _sims():
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        dev = FDTD(span(N[0], D), span(N[1], D), span(N[2], D), D, D, D, 1.55)
    host = types.SimpleNamespace(Nx=N[0], Ny=N[1], Nz=N[2], YEE_SHIFTS=FDTD.YEE_SHIFTS)
    return dev, host


def _same(eps, prim, velocity, **kw):
    dev, host = _sims()
    a = boundary_deps(dev, eps, prim, velocity, **kw)
    b = boundary_deps(host, eps, prim, velocity, **kw)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and np.array_equal(x, y)
    return len(a[0])


@pytest.mark.parametrize("seed", [0, 1, 2, 5])
def test_device_derivatives_match_host(seed):
    rng = np.random.default_rng(seed)
    X, Y, Z = (n * D for n in N)
    eps = StructuredMaterial3D(X, Y, Z, D, D, D, background=2.07 + 0.1j * (seed % 2),
                               ellipse_vertices=20)
    prims = []
    for q in range(6):
        val, layer = complex(2 + 10 * rng.random(), 0.2 * rng.random() * (q % 2)), int(rng.integers(1, 5))
        x, y = rng.uniform(0, X), rng.uniform(0, Y)
        if q % 3 == 0:
            w, h = rng.uniform(0.1, 0.6, 2)
            if q == 0:
                x, y, w, h = 10 * D, 8 * D, 8 * D, 6 * D      # on cell boundaries
            p = Rectangle(x, y, w, h, material_value=val, layer=layer)
        elif q % 3 == 1:
            n = int(rng.integers(3, 70 if q == 4 else 9))
            ang, r = np.sort(rng.uniform(0, 2 * np.pi, n)), rng.uniform(0.05, 0.4, n)
            p = Polygon(x + r * np.cos(ang), y + r * np.sin(ang), material_value=val, layer=layer)
        else:
            p = Ellipse(x, y, *rng.uniform(0.1, 0.4, 2), rng.uniform(0, np.pi), material_value=val,
                        layer=layer)
        z1 = rng.uniform(-0.1, 0.3)
        eps.add_primitive(p, z1, z1 + rng.uniform(0.05, 0.4))
        prims.append(p)
    found = 0
    print(seed, flush=True)
    for p in prims:
        if isinstance(p, Rectangle):
            found += sum(_same(eps, p, rect_edge_velocity(e), tol=1e-3 * (seed % 2))
                         for e in ("xl", "yt"))
        elif isinstance(p, Polygon):
            n = len(p.xs)
            found += _same(eps, p, polygon_vertex_velocity(n, n // 2, (0.6, -0.8)))
            found += _same(eps, p, rng.standard_normal((n, 2)))
    assert found > 0


def test_more_primitives_than_the_device_holds():
    eps = StructuredMaterial3D(1.0, 0.85, 0.4, D, D, D)
    for q in range(10):
        r = Rectangle(0.5, 0.4, 0.4 + 1e-3 * q, 0.3 + 1e-3 * q, material_value=2.0 + q, layer=q + 1)
        eps.add_primitive(r, 0.0, 0.4)
    assert _same(eps, r, rect_edge_velocity("xr")) > 0
