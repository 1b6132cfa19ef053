"""Material distributions for the solver (host side, numpy).

The solver only needs an object with ``get_values(k1, k2, j1, j2, i1, i2, sx,
sy, sz, arr)`` returning complex values on the (shifted) Yee grid, the
interface of ``emopt.grid.Material3D`` (emopt/grid.py:723-845).  This module
provides:

* :class:`ConstantMaterial3D` (emopt/grid.py:846-872)
* :class:`StructuredMaterial3D` -- z-stacked primitives with layer priority
  and cell averaging (emopt/grid.py:874-961, src/Grid.cpp:460-525,736-874)
* primitives :class:`Rectangle`, :class:`Polygon`, :class:`Ellipse`
* :class:`FunctionMaterial3D` for analytic / array-backed distributions.

StructuredMaterial3D also samples on the GPU (``get_values_device``, the
emf_sample_structured kernels), with the arithmetic below operation for
operation; FDTD.build/update use that path for it.

Cell averaging: a Yee cell value is the sum over z-slabs of the stack of
(slab fraction of the cell's z extent) x (in-plane average), background 1.0
outside the stack, exactly as src/Grid.cpp:736-824 combines layers.  The
in-plane average follows one of two rules:

* ``overlap="exact"`` (default), the reference's rule
  (StructuredMaterial2D::get_value, src/Grid.cpp:460-525): primitives are
  visited in priority order (lower ``layer`` first); one counts in a cell only
  when a cell corner lies strictly inside it; if all four corners are inside
  and nothing of the cell is taken yet the cell takes its value; otherwise it
  takes the exact area of the part of the cell not yet taken that it covers
  (GridCell::intersect, src/Grid.cpp:74-108, boost.geometry in __float128
  there, a slab sweep in double precision here); the cell stops once nothing
  is left, and the rest is background.  Ellipses (which the reference builds
  as polygons) are inscribed polygons of ``ellipse_vertices`` vertices.
* ``overlap="supersample"``: each primitive takes min(coverage, what is left);
  rectangle coverage is exact, ellipse and polygon coverage is the fraction of
  ``supersample`` x ``supersample`` points inside.
"""
from __future__ import annotations

import numpy as np


class Material3D:
    def get_value(self, x, y, z):
        v = self.get_values(0, 1, 0, 1, 0, 1, sx=x, sy=y, sz=z)
        return v.ravel()[0]

    def get_values(self, k1, k2, j1, j2, i1, i2, sx=0.0, sy=0.0, sz=0.0, arr=None, reshape=True):
        raise NotImplementedError

    def get_values_in(self, domain, sx=0.0, sy=0.0, sz=0.0, arr=None, squeeze=False):
        v = self.get_values(domain.k1, domain.k2, domain.j1, domain.j2, domain.i1, domain.i2,
                            sx, sy, sz, arr)
        return np.squeeze(v) if squeeze else v

    @staticmethod
    def _out(vals, arr, reshape):
        if arr is not None:
            flat = np.ravel(arr)
            flat[:] = vals.ravel()
            vals = flat if not reshape else flat.reshape(vals.shape)
        return vals if reshape else vals.ravel()


class ConstantMaterial3D(Material3D):
    def __init__(self, value):
        self._value = complex(value)

    @property
    def material_value(self):
        return self._value

    @material_value.setter
    def material_value(self, v):
        self._value = complex(v)

    def get_values(self, k1, k2, j1, j2, i1, i2, sx=0.0, sy=0.0, sz=0.0, arr=None, reshape=True):
        vals = np.full((i2 - i1, j2 - j1, k2 - k1), self._value, dtype=np.complex128)
        return self._out(vals, arr, reshape)


class FunctionMaterial3D(Material3D):
    """Values from ``func(x, y, z)`` evaluated at the Yee-shifted cell
    positions (x = (k + sx) * dx etc.), broadcast over [Nz, Ny, Nx]."""

    def __init__(self, func, dx, dy, dz):
        self._f = func
        self._d = (dx, dy, dz)

    def get_values(self, k1, k2, j1, j2, i1, i2, sx=0.0, sy=0.0, sz=0.0, arr=None, reshape=True):
        dx, dy, dz = self._d
        x = (np.arange(k1, k2) + sx) * dx
        y = (np.arange(j1, j2) + sy) * dy
        z = (np.arange(i1, i2) + sz) * dz
        Z, Y, X = np.meshgrid(z, y, x, indexing="ij")
        vals = np.asarray(self._f(X, Y, Z), dtype=np.complex128)
        vals = np.broadcast_to(vals, (i2 - i1, j2 - j1, k2 - k1)).copy()
        return self._out(vals, arr, reshape)


class GridMaterial3D(Material3D):
    """Values held in an array ``grid[i, j, k]`` over an Nx x Ny x Nz grid of
    size X x Y x Z (emopt/grid.py:238-251).  get_values returns the cells of
    a box as they are, for every Yee offset."""

    def __init__(self, X, Y, Z, Nx, Ny, Nz, grid):
        self.X, self.Y, self.Z = X, Y, Z
        self.Nx, self.Ny, self.Nz = Nx, Ny, Nz
        self.grid = grid

    def get_value(self, k, j, i):
        return self.grid[i, j, k]

    def get_values(self, k1, k2, j1, j2, i1, i2, sx=0.0, sy=0.0, sz=0.0, arr=None, reshape=True):
        vals = np.asarray(self.grid, dtype=np.complex128)[i1:i2, j1:j2, k1:k2].copy()
        return self._out(vals, arr, reshape)


# ------------------------------------------------------------- primitives

class MaterialPrimitive:
    def __init__(self, material_value=1.0, layer=1):
        self.material_value = complex(material_value)
        self.layer = layer

    def set_material(self, mat):
        self.material_value = complex(mat)

    # the deprecated accessors of emopt/grid.py:288-310
    def get_layer(self):
        return self.layer

    def set_layer(self, layer):
        self.layer = layer

    def contains_point(self, x, y):
        """True when (x, y) lies strictly inside the primitive, the test the
        overlap rule applies to cell corners (emopt/grid.py:312-328)."""
        inside = StructuredMaterial3D._ring_of(self, 128)
        if inside is None:
            return False
        return bool(inside.within(np.asarray([float(x)]), np.asarray([float(y)]))[0])

    def coverage(self, xc, yc, dx, dy, ss):
        """Area fraction of each cell centred at (yc[:,None], xc[None,:]) of
        size dx*dy covered by the primitive, shape [len(yc), len(xc)]."""
        raise NotImplementedError

    def bbox(self):
        raise NotImplementedError


class Rectangle(MaterialPrimitive):
    """Axis-aligned rectangle centred at (x0, y0) (emopt/grid.py:367-501)."""

    def __init__(self, x0, y0, xspan, yspan, material_value=1.0, layer=1):
        super().__init__(material_value, layer)
        self.x0, self.y0, self.width, self.height = x0, y0, xspan, yspan

    # the setters of emopt/grid.py:465-501
    def set_position(self, x0, y0):
        self.x0, self.y0 = x0, y0

    def set_width(self, width):
        self.width = width

    def set_height(self, height):
        self.height = height

    def bbox(self):
        return (self.x0 - self.width / 2, self.x0 + self.width / 2,
                self.y0 - self.height / 2, self.y0 + self.height / 2)

    def coverage(self, xc, yc, dx, dy, ss):
        x0, x1, y0, y1 = self.bbox()
        fx = np.clip(np.minimum(xc + dx / 2, x1) - np.maximum(xc - dx / 2, x0), 0, None) / dx
        fy = np.clip(np.minimum(yc + dy / 2, y1) - np.maximum(yc - dy / 2, y0), 0, None) / dy
        return fy[:, None] * fx[None, :]

    def ring(self):
        """The polygon ring of src/Grid.cpp:204-213."""
        x0, x1, y0, y1 = self.bbox()
        return np.array([x0, x0, x1, x1]), np.array([y0, y1, y1, y0])


class _Sampled(MaterialPrimitive):
    def inside(self, x, y):
        raise NotImplementedError

    def coverage(self, xc, yc, dx, dy, ss):
        out = np.zeros((len(yc), len(xc)))
        xb0, xb1, yb0, yb1 = self.bbox()
        kx = np.nonzero((xc + dx / 2 > xb0) & (xc - dx / 2 < xb1))[0]
        ky = np.nonzero((yc + dy / 2 > yb0) & (yc - dy / 2 < yb1))[0]
        if len(kx) == 0 or len(ky) == 0:
            return out
        off = (np.arange(ss) + 0.5) / ss - 0.5
        xs = (xc[kx][:, None] + off[None, :] * dx).ravel()
        ys = (yc[ky][:, None] + off[None, :] * dy).ravel()
        Y, X = np.meshgrid(ys, xs, indexing="ij")
        ins = self.inside(X, Y).astype(np.float64)
        ins = ins.reshape(len(ky), ss, len(kx), ss).mean(axis=(1, 3))
        out[np.ix_(ky, kx)] = ins
        return out


class Ellipse(_Sampled):
    """Ellipse centred at (x0, y0) with semi-axes (a, b), rotated by angle,
    optionally clipped to the box clip = (xmin, xmax, ymin, ymax)."""

    def __init__(self, x0, y0, a, b, angle=0.0, material_value=1.0, layer=1, clip=None):
        super().__init__(material_value, layer)
        self.x0, self.y0, self.a, self.b, self.angle = x0, y0, a, b, angle
        self.clip = clip

    def bbox(self):
        r = max(self.a, self.b)
        x0, x1, y0, y1 = self.x0 - r, self.x0 + r, self.y0 - r, self.y0 + r
        if self.clip is not None:
            x0, x1 = max(x0, self.clip[0]), min(x1, self.clip[1])
            y0, y1 = max(y0, self.clip[2]), min(y1, self.clip[3])
        return x0, x1, y0, y1

    def polygon(self, n):
        """Vertices of the inscribed n-gon (points at angles 2 pi i / n of the
        ellipse's own axes), clipped to the clip box; empty arrays when
        nothing is left."""
        t = 2 * np.pi * np.arange(n) / n
        u, v = self.a * np.cos(t), self.b * np.sin(t)
        c, s = np.cos(self.angle), np.sin(self.angle)
        xs, ys = self.x0 + u * c - v * s, self.y0 + u * s + v * c
        if self.clip is not None:
            xs, ys = _clip_to_box(xs, ys, self.clip)
        return xs, ys

    def inside(self, x, y):
        c, s = np.cos(self.angle), np.sin(self.angle)
        u = (x - self.x0) * c + (y - self.y0) * s
        v = -(x - self.x0) * s + (y - self.y0) * c
        ins = (u / self.a) ** 2 + (v / self.b) ** 2 <= 1.0
        if self.clip is not None:
            ins &= (x >= self.clip[0]) & (x < self.clip[1]) & (y >= self.clip[2]) & (y < self.clip[3])
        return ins


class Polygon(_Sampled):
    """Simple polygon from vertex lists (emopt/grid.py:503-651); even-odd rule."""

    def __init__(self, xs=None, ys=None, material_value=1.0, layer=1):
        super().__init__(material_value, layer)
        self.xs = np.asarray(xs if xs is not None else [], dtype=np.double)
        self.ys = np.asarray(ys if ys is not None else [], dtype=np.double)

    def set_points(self, xs, ys):
        self.xs = np.asarray(xs, dtype=np.double)
        self.ys = np.asarray(ys, dtype=np.double)

    # vertex editing of emopt/grid.py:556-592
    @property
    def Np(self):
        return len(self.xs)

    def add_point(self, x, y):
        self.xs = np.append(self.xs, float(x))
        self.ys = np.append(self.ys, float(y))

    def add_points(self, x, y):
        self.xs = np.concatenate([self.xs, np.asarray(x, dtype=np.double)])
        self.ys = np.concatenate([self.ys, np.asarray(y, dtype=np.double)])

    def set_point(self, index, x, y):
        self.xs = np.array(self.xs, dtype=np.double)
        self.ys = np.array(self.ys, dtype=np.double)
        self.xs[index], self.ys[index] = x, y

    @staticmethod
    def populate_lines(xs, ys, ds):
        """Points spaced at least ds along the connected segments (xs,
        ys): a segment of length s is cut into max(ceil(s / ds), 2) - 1
        equal pieces, its far end kept (emopt/grid.py:594-651)."""
        outx, outy = [np.asarray([xs[0]], dtype=np.double)], [np.asarray([ys[0]], dtype=np.double)]
        for a in range(len(xs) - 1):
            n = max(int(np.ceil(np.hypot(xs[a + 1] - xs[a], ys[a + 1] - ys[a]) / ds)), 2)
            outx.append(np.linspace(xs[a], xs[a + 1], n)[1:])
            outy.append(np.linspace(ys[a], ys[a + 1], n)[1:])
        return np.concatenate(outx), np.concatenate(outy)

    def bbox(self):
        return self.xs.min(), self.xs.max(), self.ys.min(), self.ys.max()

    def ring(self):
        return self.xs, self.ys

    def inside(self, x, y):
        res = np.zeros(x.shape, dtype=bool)
        xs, ys = self.xs, self.ys
        n = len(xs)
        for a in range(n):
            b = (a + 1) % n
            xa, ya, xb, yb = xs[a], ys[a], xs[b], ys[b]
            if ya == yb:
                continue
            cond = (ya > y) != (yb > y)
            xint = xa + (y - ya) * (xb - xa) / (yb - ya)
            res ^= cond & (x < xint)
        return res


def _clip_to_box(xs, ys, box):
    """Sutherland-Hodgman clip of a polygon to an axis-aligned box."""
    if len(xs) >= 3 and min(xs) >= box[0] and max(xs) <= box[1] and min(ys) >= box[2] \
            and max(ys) <= box[3]:
        return np.array(xs), np.array(ys)        # inside: as it is
    pts = list(zip(xs, ys))
    for axis, val, keep_above in ((0, box[0], True), (0, box[1], False),
                                  (1, box[2], True), (1, box[3], False)):
        if not pts:
            break
        out = []
        for a in range(len(pts)):
            p, q = pts[a - 1], pts[a]
            pin = p[axis] >= val if keep_above else p[axis] <= val
            qin = q[axis] >= val if keep_above else q[axis] <= val
            if pin != qin:
                t = (val - p[axis]) / (q[axis] - p[axis])
                cut = [p[0] + t * (q[0] - p[0]), p[1] + t * (q[1] - p[1])]
                cut[axis] = val
                out.append(tuple(cut))
            if qin:
                out.append(q)
        pts = out
    if len(pts) < 3:
        return np.zeros(0), np.zeros(0)
    return np.array([p[0] for p in pts]), np.array([p[1] for p in pts])


# ------------------------------------------- the reference's overlap rule
# Limits of one cell, as in the device sampler (emf_sample_structured).
_MAXU, _MAXE, _MAXB = 8, 48, 256


class _Ring:
    """A rectangle (kind 0) or polygon (kind 2) as the exact rule sees it."""

    def __init__(self, kind, xs, ys, bbox, value):
        self.kind, self.xs, self.ys = kind, np.asarray(xs, float), np.asarray(ys, float)
        self.bbox = tuple(float(b) for b in bbox)
        self.value = complex(value)

    def within(self, x, y):
        """Strictly inside, elementwise (boundary points are out: boost's
        within, src/Grid.cpp:362-374; Rectangle::contains_point,
        src/Grid.cpp:219-225)."""
        b = self.bbox
        res = (x > b[0]) & (x < b[1]) & (y > b[2]) & (y < b[3])
        if self.kind == 0 or not np.any(res):
            return res
        odd = np.zeros(np.shape(x), dtype=bool)
        edge = np.zeros(np.shape(x), dtype=bool)
        xs, ys = self.xs, self.ys
        n = len(xs)
        for a in range(n):
            c = a + 1 if a + 1 < n else 0
            xa, ya, xb, yb = xs[a], ys[a], xs[c], ys[c]
            edge |= (((xb - xa) * (y - ya) - (yb - ya) * (x - xa) == 0.0) &
                     (x >= min(xa, xb)) & (x <= max(xa, xb)) & (y >= min(ya, yb)) & (y <= max(ya, yb)))
            if (ya > yb) or (ya < yb):
                with np.errstate(divide="ignore", invalid="ignore"):
                    xint = xa + (y - ya) * (xb - xa) / (yb - ya)
                odd ^= ((ya > y) != (yb > y)) & (x < xint)
        return res & odd & ~edge


def _union_area(rings, xa, xb, ya, yb):
    """Area of [xa, xb] x [ya, yb] inside the union of the rings: between
    consecutive x breakpoints (ends of the edges through the cell, their
    crossings of y = ya and y = yb, crossings of edges of different rings
    inside the cell) the covered length of a vertical line is linear, so each
    slab adds width x covered length at its midpoint; the line enters the
    cell inside a ring when an odd number of the ring's edges cross it at or
    below ya.  The operations are those of mat_union_area in
    emopt_amd/csrc/material.hpp, in the same order."""
    e = []
    for q, r in enumerate(rings):
        xs, ys = r.xs, r.ys
        nxt = np.r_[np.arange(1, len(xs)), 0]
        x2, y2 = xs[nxt], ys[nxt]
        keep = ~((np.maximum(xs, x2) <= xa) | (np.minimum(xs, x2) >= xb) |
                 (np.maximum(ys, y2) <= ya) | (np.minimum(ys, y2) >= yb))
        for a in np.nonzero(keep)[0]:
            if len(e) == _MAXE:
                raise ValueError(_LIMIT_MSG)
            e.append((float(xs[a]), float(ys[a]), float(x2[a]), float(y2[a]), q))
    bx = [xa, xb]

    def push(x):
        if not (x > xa and x < xb):
            return
        if len(bx) == _MAXB:
            raise ValueError(_LIMIT_MSG)
        bx.append(x)

    for x1, y1, x2, y2, _ in e:
        push(x1)
        push(x2)
        if (y1 > ya) != (y2 > ya):
            push(x1 + (ya - y1) * (x2 - x1) / (y2 - y1))
        if (y1 > yb) != (y2 > yb):
            push(x1 + (yb - y1) * (x2 - x1) / (y2 - y1))
    for i in range(len(e)):
        fx1, fy1, fx2, fy2, fq = e[i]
        for j in range(i + 1, len(e)):
            hx1, hy1, hx2, hy2, hq = e[j]
            if fq == hq:
                continue
            d = (fx2 - fx1) * (hy2 - hy1) - (fy2 - fy1) * (hx2 - hx1)
            if d == 0.0:
                continue
            t = ((hx1 - fx1) * (hy2 - hy1) - (hy1 - fy1) * (hx2 - hx1)) / d
            r = ((hx1 - fx1) * (fy2 - fy1) - (hy1 - fy1) * (fx2 - fx1)) / d
            if not (t > 0.0 and t < 1.0 and r > 0.0 and r < 1.0):
                continue
            y = fy1 + t * (fy2 - fy1)
            if y > ya and y < yb:
                push(fx1 + t * (fx2 - fx1))
    bx.sort()
    rx = []
    for r in rings:
        nxt = np.r_[np.arange(1, len(r.xs)), 0]
        rx.append((r.xs, r.ys, r.xs[nxt], r.ys[nxt]))
    area = 0.0
    for b in range(len(bx) - 1):
        w = bx[b + 1] - bx[b]
        if not w > 0.0:
            continue
        xm = 0.5 * (bx[b] + bx[b + 1])
        inside = 0
        for q, (x1, y1, x2, y2) in enumerate(rx):
            cross = (np.minimum(x1, x2) < xm) & (np.maximum(x1, x2) > xm)
            with np.errstate(divide="ignore", invalid="ignore"):
                y = y1 + (xm - x1) * (y2 - y1) / (x2 - x1)
            if np.count_nonzero(cross & (y <= ya)) % 2:
                inside ^= 1 << q
        ev = []
        for x1, y1, x2, y2, q in e:
            if not (min(x1, x2) < xm and max(x1, x2) > xm):
                continue
            y = y1 + (xm - x1) * (y2 - y1) / (x2 - x1)
            if y > ya and y < yb:
                ev.append((y, q))
        ev.sort(key=lambda v: v[0])
        length, yp = 0.0, ya
        for y, q in ev:
            if inside:
                length += y - yp
            yp = y
            inside ^= 1 << q
        if inside:
            length += yb - yp
        area += w * length
    return area


_LIMIT_MSG = ("a cell meets more than %d primitives or %d polygon edges "
              "(exact overlap rule)" % (_MAXU, _MAXE))


def _cell_exact(order, xa, xb, ya, yb, bg):
    """One cell by the reference's rule, the operations of k_mat_exact
    in the same order; order = the rings' corner flags
    (c1, c2, c3, c4) in priority order."""
    A = (xb - xa) * (yb - ya)
    rem = A
    vr = vi = 0.0
    used = []
    for r, (c1, c2, c3, c4) in order:
        if c1 and c2 and c3 and c4 and rem == A:
            return r.value.real, r.value.imag
        if c1 or c2 or c3 or c4:
            if len(used) == _MAXU:
                raise ValueError(_LIMIT_MSG)
            used.append(r)
            rn = A - _union_area(used, xa, xb, ya, yb)
            if rn <= A * 1e-13:
                rn = 0.0
            ov = (rem - rn) / A
            vr += ov * r.value.real
            vi += ov * r.value.imag
            rem = rn
        if rem == 0.0:
            break
    if rem > 0.0:
        f = rem / A
        vr += f * bg.real
        vi += f * bg.imag
    return vr, vi


class StructuredMaterial3D(Material3D):
    """Primitives extruded over [z1, z2) ranges (emopt/grid.py:874-961)."""

    def __init__(self, X, Y, Z, dx, dy, dz, supersample=8, background=1.0, overlap="exact",
                 ellipse_vertices=128):
        if overlap not in ("exact", "supersample"):
            raise ValueError("overlap must be 'exact' or 'supersample'")
        self._X, self._Y, self._Z = X, Y, Z
        self._dx, self._dy, self._dz = dx, dy, dz
        self.supersample = supersample
        self.background = complex(background)
        self.overlap = overlap
        self.ellipse_vertices = int(ellipse_vertices)
        self._prims = []    # (prim, z1, z2, insertion order)

    @property
    def primitives(self):
        return [p for p, _, _, _ in self._prims]

    def add_primitive(self, prim, z1, z2):
        if z2 <= z1:
            return
        self._prims.append((prim, float(z1), float(z2), len(self._prims)))

    def add_primitives(self, prims, z1, z2):
        for p in prims:
            self.add_primitive(p, z1, z2)

    @property
    def zmins(self):
        return [z1 for _, z1, _, _ in self._prims]

    @property
    def zmaxs(self):
        return [z2 for _, _, z2, _ in self._prims]

    def _ring(self, prim):
        return self._ring_of(prim, self.ellipse_vertices)

    @staticmethod
    def _ring_of(prim, ellipse_vertices):
        """The primitive as the exact rule sees it (None: nothing left)."""
        if isinstance(prim, Rectangle):
            return _Ring(0, *prim.ring(), prim.bbox(), prim.material_value)
        if isinstance(prim, Ellipse):
            xs, ys = prim.polygon(ellipse_vertices)
        elif isinstance(prim, Polygon):
            xs, ys = prim.ring()
        else:
            raise TypeError("no overlap rule for %s" % type(prim).__name__)
        if len(xs) < 3:
            return None
        return _Ring(2, xs, ys, (xs.min(), xs.max(), ys.min(), ys.max()), prim.material_value)

    def _inplane_exact(self, active, xc, yc):
        dx, dy = self._dx, self._dy
        rings = [r for r in (self._ring(p[0]) for p in sorted(active, key=lambda p: (p[0].layer, p[3])))
                 if r is not None]
        xa, xb = xc - dx / 2, xc + dx / 2
        ya, yb = yc - dy / 2, yc + dy / 2
        ny, nx = len(yc), len(xc)
        bg = self.background
        vr = np.full((ny, nx), 1.0 * bg.real)
        vi = np.full((ny, nx), 1.0 * bg.imag)
        flags = []
        decided = np.zeros((ny, nx), dtype=bool)
        partial = np.zeros((ny, nx), dtype=bool)
        for r in rings:
            c = [np.zeros((ny, nx), dtype=bool) for _ in range(4)]
            kx = np.nonzero((xb > r.bbox[0]) & (xa < r.bbox[1]))[0]
            ky = np.nonzero((yb > r.bbox[2]) & (ya < r.bbox[3]))[0]
            if len(kx) and len(ky):
                blk = np.ix_(ky, kx)
                XA, YA = np.meshgrid(xa[kx], ya[ky])
                XB, YB = np.meshgrid(xb[kx], yb[ky])
                for q, (X, Y) in enumerate(((XA, YA), (XB, YA), (XB, YB), (XA, YB))):
                    c[q][blk] = r.within(X, Y)
            flags.append(c)
            anyc = c[0] | c[1] | c[2] | c[3]
            allc = c[0] & c[1] & c[2] & c[3]
            first = anyc & ~decided
            full = first & allc
            vr[full] = r.value.real
            vi[full] = r.value.imag
            partial |= first & ~allc
            decided |= first
        for j, k in zip(*np.nonzero(partial)):
            order = [(r, tuple(bool(f[q][j, k]) for q in range(4))) for r, f in zip(rings, flags)]
            vr[j, k], vi[j, k] = _cell_exact(order, xa[k], xb[k], ya[j], yb[j], bg)
        out = np.empty((ny, nx), dtype=np.complex128)
        out.real, out.imag = vr, vi
        return out

    def _inplane(self, active, xc, yc):
        if self.overlap == "exact":
            return self._inplane_exact(active, xc, yc)
        dx, dy = self._dx, self._dy
        remaining = np.ones((len(yc), len(xc)))
        val = np.zeros((len(yc), len(xc)), dtype=np.complex128)
        for prim in sorted(active, key=lambda p: (p[0].layer, p[3])):
            cov = np.minimum(prim[0].coverage(xc, yc, dx, dy, self.supersample), remaining)
            val += cov * prim[0].material_value
            remaining -= cov
        val += remaining * self.background
        return val

    # emf_prim of include/emfdtd.h
    PRIM_DTYPE = np.dtype([("kind", "<i4"), ("clip", "<i4"), ("v0", "<i4"), ("nv", "<i4"),
                           ("re", "<f8"), ("im", "<f8"), ("z1", "<f8"), ("z2", "<f8"),
                           ("bbox", "<f8", (4,)), ("q", "<f8", (10,))])

    def device_primitives(self):
        """The primitives as emf_prim records in priority order (layer, then
        insertion), with the polygon vertex arrays.  Under the exact rule an
        ellipse goes as its inscribed polygon (and one clipped to nothing is
        left out)."""
        order = sorted(self._prims, key=lambda p: (p[0].layer, p[3]))
        if self.overlap == "exact":
            order = [(p if not isinstance(p, Ellipse) else self._ring(p), z1, z2, n)
                     for p, z1, z2, n in order]
            order = [o for o in order if o[0] is not None]
        recs = np.zeros(len(order), dtype=self.PRIM_DTYPE)
        vx, vy = [], []
        nv = 0
        for r, (prim, z1, z2, _) in zip(recs, order):
            r["z1"], r["z2"] = z1, z2
            if isinstance(prim, _Ring):       # an ellipse as a polygon
                r["re"], r["im"] = prim.value.real, prim.value.imag
                r["bbox"] = prim.bbox
                r["kind"] = 2
                r["v0"], r["nv"] = nv, len(prim.xs)
                vx.append(prim.xs)
                vy.append(prim.ys)
                nv += len(prim.xs)
                continue
            r["re"], r["im"] = prim.material_value.real, prim.material_value.imag
            r["bbox"] = prim.bbox()
            if isinstance(prim, Rectangle):
                r["kind"] = 0
            elif isinstance(prim, Ellipse):
                r["kind"] = 1
                r["q"][:6] = (prim.x0, prim.y0, prim.a, prim.b, np.cos(prim.angle), np.sin(prim.angle))
                if prim.clip is not None:
                    r["clip"] = 1
                    r["q"][6:] = prim.clip
            elif isinstance(prim, Polygon):
                r["kind"] = 2
                r["v0"], r["nv"] = nv, len(prim.xs)
                vx.append(prim.xs)
                vy.append(prim.ys)
                nv += len(prim.xs)
            else:
                raise TypeError("no device sampler for %s" % type(prim).__name__)
        vx = np.ascontiguousarray(np.concatenate(vx) if vx else np.zeros(1), dtype=np.double)
        vy = np.ascontiguousarray(np.concatenate(vy) if vy else np.zeros(1), dtype=np.double)
        return recs, vx, vy, nv

    def get_values_device(self, k1, k2, j1, j2, i1, i2, sx=0.0, sy=0.0, sz=0.0, device=0,
                          arr=None, reshape=True):
        """get_values computed on GPU `device` (emf_sample_structured): the
        same arithmetic in the same order, so the same doubles."""
        from . import _lib
        lib = _lib.load()
        recs, vx, vy, nv = self.device_primitives()
        out = np.empty((i2 - i1, j2 - j1, k2 - k1), dtype=np.complex128)
        lib.emf_sample_structured(int(device), recs.ctypes.data, len(recs), vx.ctypes.data,
                                  vy.ctypes.data, nv, self._dx, self._dy, self._dz,
                                  0 if self.overlap == "exact" else int(self.supersample),
                                  self.background.real, self.background.imag,
                                  k1, k2, j1, j2, i1, i2, sx, sy, sz, out.ctypes.data)
        return self._out(out, arr, reshape)

    def stock_samplers(self):
        """Whether get_values and get_values_device are this module's own."""
        return all(getattr(getattr(self, f), "__func__", None) is fn
                   for f, fn in _STOCK_SAMPLERS.items())

    def build_device(self, lib, handle, shifts, mu):
        """Sample eps at three in-cell offsets straight into a solver's arrays
        (emf_build_structured), with the uniform mu `mu`."""
        recs, vx, vy, nv = self.device_primitives()
        sh = np.ascontiguousarray(shifts, dtype=np.double)
        lib.emf_build_structured(handle, recs.ctypes.data, len(recs), vx.ctypes.data,
                                 vy.ctypes.data, nv, self._dx, self._dy, self._dz,
                                 0 if self.overlap == "exact" else int(self.supersample),
                                 self.background.real, self.background.imag, sh.ctypes.data,
                                 float(mu))

    def get_values(self, k1, k2, j1, j2, i1, i2, sx=0.0, sy=0.0, sz=0.0, arr=None, reshape=True):
        dx, dy, dz = self._dx, self._dy, self._dz
        xc = (np.arange(k1, k2) + sx) * dx
        yc = (np.arange(j1, j2) + sy) * dy
        zc = (np.arange(i1, i2) + sz) * dz
        zlo, zhi = zc - dz / 2, zc + dz / 2
        out = np.zeros((i2 - i1, j2 - j1, k2 - k1), dtype=np.complex128)
        covered = np.zeros(i2 - i1)
        prims = self._prims
        if self.overlap == "exact":    # as device_primitives: no ellipse clipped to nothing
            prims = [p for p in prims if not isinstance(p[0], Ellipse) or self._ring(p[0]) is not None]
        bounds = sorted({b for _, z1, z2, _ in prims for b in (z1, z2)})
        for za, zb in zip(bounds[:-1], bounds[1:]):
            fz = np.clip(np.minimum(zhi, zb) - np.maximum(zlo, za), 0, None) / dz
            if not np.any(fz > 0):
                continue
            active = [p for p in prims if p[1] <= za and p[2] >= zb]
            v2 = self._inplane(active, xc, yc)
            nz = np.nonzero(fz > 0)[0]
            out[nz] += fz[nz, None, None] * v2[None, :, :]
            covered += fz
        out += (1.0 - covered)[:, None, None] * self.background
        return self._out(out, arr, reshape)


_STOCK_SAMPLERS = {"get_values": StructuredMaterial3D.get_values,
                   "get_values_device": StructuredMaterial3D.get_values_device}
