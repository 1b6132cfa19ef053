"""Performance cases of the CW-FDTD framework: the calls a design script makes, from the
smallest test grid to a 400x200x120 solve.

Six kinds of case:

* ``solve``     FDTD.solve_forward and the download of the solved fields,
* ``batch``     a Batch of forward and adjoint solves of different sizes,
* ``gradient``  figure of merit and gradient of an adjoint method (forward solve, adjoint
                sources, adjoint solve, gradient assembly),
* ``build``     FDTD.build of a structured material and get_A_diag,
* ``fields``    interpolated monitor planes and the source power of a solved problem,
* ``assemble``  sparse gradient assembly and y^T dA x over a box.

A solve runs to convergence (``steps`` = 0) or a fixed number of steps, as parity runs and
finite-difference checks do.  ``exact`` is a plain torch float64 time stepper of the same
problem (leapfrog updates, CPML, sources, convergence check, three-sample phasors).
"""
import math
import warnings

import numpy as np
import torch

from emopt_amd.adjoint import AdjointMethodPNF3D, ModeMatch
from emopt_amd.batch import Batch
from emopt_amd.fdtd import FDTD
from emopt_amd.grid import ConstantMaterial3D, Ellipse, Rectangle, StructuredMaterial3D
from emopt_amd.misc import DomainCoordinates, gaussian_mode
from emopt_amd.shape import boundary_deps, rect_edge_velocity

EPS_SI, EPS_OX = 3.48 ** 2, 1.444 ** 2
COMPS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")
# positions of eps_x, eps_y, eps_z, mu_x, mu_y, mu_z within a cell
YEE = ((0.5, 0.0, -0.5), (0.0, 0.5, -0.5), (0.0, 0.0, 0.0),
       (0.0, 0.5, 0.0), (0.5, 0.0, 0.0), (0.5, 0.5, -0.5))


def _case(name, kind, Nx, Ny, Nz, **kw):
    c = dict(name=name, kind=kind, Nx=Nx, Ny=Ny, Nz=Nz, d=0.04, wl=1.55, pml=10, bc="000",
             device="strip", loss=0.0, mu=1.0, steps=0, nconv=10, members=1)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest solve: a quick check of a script, where launches and latency count
        _case("solve_24x20x16", "solve", 24, 20, 16, pml=4),
        # a cubic cell of a parameter sweep, the low end of what a solve server receives
        _case("solve_64x64x64", "solve", 64, 64, 64, device="ellipses", steps=900),
        # straight strip waveguide run to convergence
        _case("solve_120x80x60", "solve", 120, 80, 60),
        # 1x2 splitter of the 3D examples: y symmetry, no CPML at the symmetry face, many
        # convergence points
        _case("solve_126x51x64_0H0", "solve", 126, 51, 64, bc="0H0", nconv=200,
              device="ellipses"),
        # a lossy device on an odd grid with a symmetry face: complex eps
        _case("solve_173x101x67_lossy", "solve", 173, 101, 67, bc="E00", loss=0.2, pml=9,
              steps=700),
        # grating-coupler sized grid
        _case("solve_360x60x120", "solve", 360, 60, 120, d=0.03, device="ellipses", steps=800),
        # the single large solve
        _case("solve_400x200x120", "solve", 400, 200, 120, d=0.03, wl=1.31, pml=12,
              device="ellipses", steps=1568),
        # forward and adjoint solves of several designs at once
        _case("batch_8", "batch", 152, 100, 68, members=8, device="ellipses", steps=500),
        # one optimiser iteration: figure of merit and its gradient
        _case("gradient_180x60x80", "gradient", 180, 60, 80, d=0.03, steps=600, members=16),
        # material sampling of a new design
        _case("build_240x120x80", "build", 240, 120, 80, d=0.03, members=40),
        # monitors of a solved problem
        _case("fields_126x76x64", "fields", 126, 76, 64, steps=160),
        # gradient from sparse material derivatives, and the box product of the gradient loop
        _case("assemble_151x126x64", "assemble", 151, 126, 64, steps=96, members=64),
    ]


def draw(rng):
    kind = rng.choice(("solve",) * 6 + ("batch", "gradient", "build", "fields", "assemble"))

    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))
    if kind == "solve":
        Nx, Ny, Nz = size(24, 400), size(20, 200), size(16, 120)
        n = Nx * Ny * Nz
        pml = min(rng.randint(4, 12), (min(Nx, Ny, Nz) - 8) // 2)
        cap = int(1.4e10 / n)          # below the largest listed solve
        steps = max(64, min(size(200, 4000), cap))
        bc = rng.choice(("000", "000", "0H0", "E00", "HE0", "00H"))
        loss = rng.choice((0.0, 0.0, 0.0, 0.2))
        mu = rng.choice((1.0, 1.0, 1.0, 1.0, 1.3))
        return _case("", kind, Nx, Ny, Nz, pml=pml, steps=steps, bc=bc, loss=loss, mu=mu,
                     wl=round(rng.uniform(1.26, 1.62), 3), d=round(rng.uniform(0.03, 0.05), 4),
                     device=rng.choice(("strip", "ellipses")))
    if kind == "batch":
        return _case("", kind, size(64, 200), size(64, 120), size(48, 72), pml=rng.randint(8, 12),
                     members=rng.randint(2, 8), steps=rng.randint(200, 600), device="ellipses")
    if kind == "gradient":
        return _case("", kind, rng.randint(140, 220), rng.randint(40, 72), 80, d=0.03,
                     steps=rng.randint(300, 700), members=2 * rng.randint(4, 9))
    if kind == "build":
        return _case("", kind, size(64, 260), size(64, 130), size(48, 90), d=0.03,
                     members=rng.randint(4, 40))
    if kind == "fields":
        return _case("", kind, size(48, 240), size(40, 130), size(40, 80), steps=160, pml=8)
    return _case("", kind, size(48, 240), size(40, 130), size(40, 80), steps=96, pml=8,
                 members=rng.randint(4, 96))


# ------------------------------------------------------------------ the problems

def _span(N, d):
    """Physical length of a grid of N points."""
    X = (N - 1) * d
    while int(np.ceil(X / d) + 1) > N:
        X = np.nextafter(X, 0.0)
    return X


def _fill(centre, d, lo, hi):
    """Covered fraction of cells of width d at `centre` by [lo, hi]."""
    return np.clip(np.minimum(centre + d / 2, hi) - np.maximum(centre - d / 2, lo), 0, None) / d


def _materials(case, rng):
    """The six sampled material arrays [Nz, Ny, Nx]: a strip waveguide along x, or a slab of
    ellipses, in cladding; lossy (complex) and magnetic cores on request."""
    Nx, Ny, Nz, d = case["Nx"], case["Ny"], case["Nz"], case["d"]
    X, Y, Z = _span(Nx, d), _span(Ny, d), _span(Nz, d)
    core = EPS_SI + 1j * case["loss"]
    width, t = rng.uniform(0.4, 0.6), rng.uniform(0.2, 0.3)
    shapes = []
    if case["device"] == "ellipses":
        for _ in range(24):
            shapes.append((rng.uniform(0.2, 0.8) * X, rng.uniform(0.2, 0.8) * Y,
                           rng.uniform(0.1, 0.6), rng.uniform(0.1, 0.6), rng.uniform(0, np.pi)))
    out = []
    for q, (sx, sy, sz) in enumerate(YEE):
        x, y, z = ((np.arange(N) + s) * d for N, s in ((Nx, sx), (Ny, sy), (Nz, sz)))
        fz = _fill(z, d, Z / 2 - t / 2, Z / 2 + t / 2)
        plane = np.broadcast_to(_fill(y, d, Y / 2 - width / 2, Y / 2 + width / 2)[:, None],
                                (Ny, Nx)).copy()
        for cx, cy, a, b, th in shapes:
            u = (x[None, :] - cx) * np.cos(th) + (y[:, None] - cy) * np.sin(th)
            v = -(x[None, :] - cx) * np.sin(th) + (y[:, None] - cy) * np.cos(th)
            r = np.sqrt((u / a) ** 2 + (v / b) ** 2)
            g = np.sqrt((u / a ** 2) ** 2 + (v / b ** 2) ** 2)
            dist = r * (r - 1) / np.maximum(g, 1e-12)      # distance to the rim, first order
            plane = np.maximum(plane, np.clip(0.5 - dist / d, 0, 1))
        f = fz[:, None, None] * plane[None]
        if q < 3:
            out.append(EPS_OX + (core - EPS_OX) * f)
        else:
            out.append((1.0 + (case["mu"] - 1.0) * f).astype(np.complex128))
    return out


def _pml(case):
    """CPML widths in cells: none on a symmetry face."""
    w = [case["pml"]] * 6
    for a in range(3):
        if case["bc"][a] in "EH":
            w[2 * a] = 0
    return w


def _source(case, rng, adjoint=False):
    """Six current arrays and their index box (k1, k2, j1, j2, i1, i2): a Gaussian line along
    y before the device, or (adjoint) a complex Gaussian on an x plane behind it."""
    Nx, Ny, Nz, d = case["Nx"], case["Ny"], case["Nz"], case["d"]
    w = _pml(case)
    y = np.arange(Ny) * d
    i = Nz // 2
    amp = rng.uniform(0.8, 1.2) * np.exp(1j * rng.uniform(0, 2 * np.pi))
    if not adjoint:
        k = min(w[0] + 5, Nx - 1)
        a = [np.zeros((1, Ny, 1), dtype=np.complex128) for _ in range(6)]
        a[2 if case["device"] == "strip" else 1][0, :, 0] = \
            amp * np.exp(-((y - y[-1] / 2) / 0.5) ** 2)
        return a, (k, k + 1, 0, Ny, i, i + 1)
    k = Nx - w[1] - 6
    J0, J1, I0, I1 = w[2] + 1, Ny - w[3] - 1, w[4] + 1, Nz - w[5] - 1
    g = np.exp(-((y[J0:J1][None, :] - y[-1] / 2) ** 2
                 + ((np.arange(I0, I1)[:, None] - i) * d) ** 2) / 0.72)
    a = [np.zeros((I1 - I0, J1 - J0, 1), dtype=np.complex128) for _ in range(6)]
    a[2][:, :, 0] = amp * g
    a[4][:, :, 0] = 0.5j * amp * g
    return a, (k, k + 1, J0, J1, I0, I1)


RAMP = 5 * 2 * np.pi
RTOL = 1e-4


def _problem(case, seed):
    """Everything a solve of `case` is made of, as arrays."""
    rng = np.random.default_rng(seed)
    return dict(mats=_materials(case, rng), fwd=_source(case, rng),
                adj=_source(case, rng, adjoint=True))


def _members(case, seed):
    """The solves of a batch: sizes around the case's, half of them adjoint."""
    rng = np.random.default_rng([9, case["members"], case["Nx"]])
    out = []
    for q in range(case["members"]):
        f = rng.uniform(0.7, 1.0, 3)
        c = dict(case, Nx=int(case["Nx"] * f[0]), Ny=int(case["Ny"] * f[1]),
                 Nz=int(case["Nz"] * f[2]), wl=float(rng.uniform(1.5, 1.6)))
        out.append((c, seed * 64 + q, q % 2 == 1))
    return out


def _solver(case, p):
    d = case["d"]
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        sim = FDTD(_span(case["Nx"], d), _span(case["Ny"], d), _span(case["Nz"], d), d, d, d,
                   case["wl"], rtol=RTOL, nconv=case["nconv"], complex_eps=case["loss"] > 0)
        sim.w_pml = [(w + 1e-9) * d for w in _pml(case)]
        sim.bc = case["bc"]
        sim.src_ramp_time = RAMP
    sim.verbose = 0
    if case["steps"]:
        sim.fixed_n0 = case["steps"]
    for (arrs, box), add in ((p["fwd"], sim.set_sources), (p["adj"], sim.add_adjoint_sources)):
        add(arrs, DomainCoordinates.from_indices(*box, d, d, d))
    sim.set_material_arrays(p["mats"][:3], p["mats"][3:])
    return sim


def _whole(case):
    return DomainCoordinates.from_indices(0, case["Nx"], 0, case["Ny"], 0, case["Nz"],
                                          case["d"], case["d"], case["d"])


def _planes(case):
    """Monitor planes (one normal to each axis) inside the CPML."""
    w, N, d = case["pml"] + 2, (case["Nx"], case["Ny"], case["Nz"]), case["d"]
    box = [[w, n - w] for n in N]
    out = []
    for a in range(3):
        b = [list(v) for v in box]
        b[a] = [N[a] // 2, N[a] // 2 + 1]
        out.append(DomainCoordinates.from_indices(*b[0], *b[1], *b[2], d, d, d))
    return out


# ------------------------------------------------------------------ prepare and run

class _Trenches(AdjointMethodPNF3D):
    """Grating of etched trenches in a slab waveguide; the parameters are their x edges."""

    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        Nx, Ny, Nz, d, w = case["Nx"], case["Ny"], case["Nz"], case["d"], case["pml"]
        X, Y, Z = _span(Nx, d), _span(Ny, d), _span(Nz, d)
        z0, etch = w * d + 0.9, 0.11
        z1 = z0 + 0.22
        eps = StructuredMaterial3D(X, Y, Z, d, d, d)
        eps.add_primitive(Rectangle(X / 2, Y / 2, 4 * X, 4 * Y, material_value=EPS_OX, layer=3),
                          -Z, z0)
        eps.add_primitive(Rectangle(X / 2, Y / 2, 4 * X, 4 * Y, material_value=EPS_SI, layer=2),
                          z0, z1)
        n = case["members"] // 2
        xs = np.linspace(w * d + 0.5, X - w * d - 0.5, n + 1)
        self.trenches, edges = [], []
        for q in range(n):
            p = xs[q + 1] - xs[q]
            a, b = xs[q] + p * rng.uniform(0.2, 0.3), xs[q] + p * rng.uniform(0.7, 0.8)
            r = Rectangle(0.5 * (a + b), Y / 2, b - a, 4 * Y, material_value=1.0, layer=1)
            eps.add_primitive(r, z1 - etch, z1)
            self.trenches.append(r)
            edges += [a, b]
        self.params = np.array(edges)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            sim = FDTD(X, Y, Z, d, d, d, case["wl"], rtol=RTOL)
            sim.w_pml = [(w + 1e-9) * d] * 6
            sim.src_ramp_time = RAMP
        sim.verbose = 0
        sim.fixed_n0 = case["steps"]
        sim.set_materials(eps, ConstantMaterial3D(1.0))
        i0, i1 = int(z0 / d) - 3, int(z1 / d) + 4
        z = np.arange(i0, i1) * d
        a = [np.zeros((i1 - i0, Ny, 1), dtype=np.complex128) for _ in range(6)]
        a[1][:, :, 0] = np.exp(-((z - 0.5 * (z0 + z1)) / 0.12) ** 2)[:, None]
        sim.set_sources(a, DomainCoordinates.from_indices(w + 3, w + 4, 0, Ny, i0, i1, d, d, d))
        self.mon = DomainCoordinates.from_indices(w + 1, Nx - w - 1, w + 1, Ny - w - 1,
                                                  Nz - w - 4, Nz - w - 3, d, d, d)
        XX, YY = np.meshgrid(self.mon.x - X / 2, self.mon.y - Y / 2)
        E, Hx, Hy = gaussian_mode(XX, YY, 3.0, 8 * np.pi / 180, case["wl"], 1.0)
        self.mm = ModeMatch([0, 0, 1], d, d, Eym=E[None], Hxm=-Hx[None], Hzm=-Hy[None])
        self.eps = eps
        super().__init__(sim, step=1e-8)

    def update_system(self, p):
        for q, r in enumerate(self.trenches):
            r.x0, r.width = 0.5 * float(p[2 * q] + p[2 * q + 1]), float(p[2 * q + 1] - p[2 * q])

    def get_fom_domains(self):
        return [self.mon]

    def calc_f(self, sim, p):
        self.mm.compute_device(sim, self.mon)
        return self.mm.get_mode_match_forward(1.0)

    def calc_dfdx_device(self, sim, p):
        self.mm.compute_device(sim, self.mon)
        return [self.mm.dFdx_device(sim, 0, mask=0b011011)]

    def calc_deps(self, sim, p):
        out = [[], [], [], []]
        for i in range(len(p)):
            comp, cell, dv = boundary_deps(sim, self.eps, self.trenches[i // 2],
                                           rect_edge_velocity("xl" if i % 2 == 0 else "xr"))
            for o, v in zip(out, (np.full(len(comp), i, np.int32), comp, cell, dv)):
                o.append(v)
        return tuple(np.concatenate(a) for a in out)


def _entries(case, rng):
    """Sparse material derivatives: 3000 cells around the core per parameter."""
    n = 3000 * case["members"]
    k, j = (rng.integers(case["pml"], N - case["pml"], n) for N in (case["Nx"], case["Ny"]))
    i = rng.integers(case["Nz"] // 2 - 4, case["Nz"] // 2 + 5, n)
    cell = (i * case["Ny"] + j) * case["Nx"] + k
    return (np.repeat(np.arange(case["members"], dtype=np.int32), 3000),
            rng.integers(0, 3, n).astype(np.int32), cell.astype(np.int64),
            rng.standard_normal(n) + 0j)


def _ydax(case, p, rng):
    """The changed diagonal of a box around the core: full arrays and the index box."""
    box = (case["Nx"] // 4, 3 * case["Nx"] // 4, case["Ny"] // 4, 3 * case["Ny"] // 4,
           case["Nz"] // 2 - 6, case["Nz"] // 2 + 6)
    k1, k2, j1, j2, i1, i2 = box
    A0 = [m.copy() for m in p["mats"][:3]]
    for a in A0:
        a[i1:i2, j1:j2, k1:k2] += 1e-3 * rng.standard_normal((i2 - i1, j2 - j1, k2 - k1))
    return A0, box


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "batch":
        s["batch"] = Batch()
        s["members"] = [(c, _solver(c, _problem(c, m)), adj)
                        for c, m, adj in _members(case, seed)]
        return s
    if kind == "gradient":
        s["am"] = _Trenches(case, seed)
        return s
    if kind == "build":
        rng = np.random.default_rng(seed)
        d = case["d"]
        X, Y, Z = (_span(case[n], d) for n in ("Nx", "Ny", "Nz"))
        eps = StructuredMaterial3D(X, Y, Z, d, d, d)
        eps.add_primitive(Rectangle(X / 2, Y / 2, 2 * X, 2 * Y, material_value=EPS_OX, layer=10),
                          -Z, 2 * Z)
        box = (0.15 * X, 0.85 * X, 0.15 * Y, 0.85 * Y)
        for _ in range(case["members"]):
            a, b = rng.uniform(0.1, 0.5, size=2)
            eps.add_primitive(Ellipse(rng.uniform(0.2, 0.8) * X, rng.uniform(0.2, 0.8) * Y, a, b,
                                      rng.uniform(0, np.pi), material_value=EPS_SI, layer=1,
                                      clip=box), Z / 2 - 0.15, Z / 2 + 0.15)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            sim = FDTD(X, Y, Z, d, d, d, case["wl"])
        sim.set_materials(eps, ConstantMaterial3D(1.0))
        s["sim"] = sim
        return s
    p = _problem(case, seed)
    s["sim"] = sim = _solver(case, p)
    if kind == "fields":
        sim.solve_forward()
    if kind == "assemble":
        rng = np.random.default_rng([3, seed])
        s["entries"] = _entries(case, rng)
        s["A0"], s["box"] = _ydax(case, p, rng)
        sim.solve_forward()
        sim.solve_adjoint()
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "solve":
        sim = state["sim"]
        sim.solve_forward()
        comps = COMPS if case["Nx"] * case["Ny"] * case["Nz"] < 2000000 else COMPS[:3]
        return [sim.get_field(c, _whole(case)) for c in comps]
    if kind == "batch":
        b = state["batch"]
        for _, sim, adj in state["members"]:
            b.add(sim, adjoint=adj)
        b.run()
        return [(sim.get_adjoint_field if adj else sim.get_field)(comp, _whole(c))
                for c, sim, adj in state["members"] for comp in COMPS[:3]]
    if kind == "gradient":
        am = state["am"]
        f = am.fom(am.params)
        return {"fom": float(f), "gradient": am.gradient_device(am.params, fom_done=True)}
    sim = state["sim"]
    if kind == "build":
        sim.build()
        return list(sim.get_A_diag())
    if kind == "fields":
        out = [sim.get_field_interp(c, p) for p in _planes(case) for c in COMPS]
        return out + [float(sim.get_source_power())]
    g = sim.grad_assemble(*state["entries"], case["members"])
    y = sim.calc_ydAx(state["A0"], box=state["box"])
    return {"gradient": g, "ydAx": np.array([y])}


def _steps(case):
    """Time steps of one solve (an estimate where it runs to convergence)."""
    tn = int(case["wl"] / case["d"] * math.sqrt(3) * 3 / 4)
    return (case["steps"] or 30 * tn) + 2 * tn


def work(case):
    """Inputs read and outputs written once; about 40 flops per cell and time step."""
    n = case["Nx"] * case["Ny"] * case["Nz"]
    kind = case["kind"]
    if kind in ("solve", "batch", "gradient"):
        cells = [n] if kind != "batch" else [c["Nx"] * c["Ny"] * c["Nz"]
                                             for c, _, _ in _members(case, 0)]
        solves = 2 if kind == "gradient" else 1
        return {"bytes": solves * sum(cells) * (3 * 16.0 + 6 * 16.0),
                "flops": solves * sum(cells) * _steps(case) * 40.0}
    if kind == "build":
        return {"bytes": n * 6 * 16.0, "flops": n * 6 * 8.0}
    if kind == "fields":
        cells = sum(int(np.prod(p.shape)) for p in _planes(case))
        return {"bytes": cells * (17 + 6) * 16.0, "flops": cells * 40.0}
    e = 3000 * case["members"]
    box = (case["Nx"] // 2) * (case["Ny"] // 2) * 12
    return {"bytes": e * (16 + 32 + 16) + box * 3 * 4 * 16.0, "flops": e * 14 + box * 3 * 16.0}


# ------------------------------------------------------------------ plain torch in 64 bits

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Axis:
    """CPML coefficients of one axis on its two slabs, and the stretched derivative
    D -> D / kappa + psi, psi <- c D + b psi."""

    def __init__(self, axis, N, w, dt, for_h, dim):
        self.parts = []
        z = axis == 2
        for side, wd in enumerate(w):
            # the first layer of the max z slab is skipped
            l = np.arange(1 if z and side == 1 else 0, wd)
            if len(l) == 0:
                continue
            if for_h:
                q = l / wd if z else (l - 0.5 if side == 0 else l + 0.5) / wd
            else:
                q = l / wd if not z else (l + 0.5 if side == 0 else l - 0.5) / wd
            f = np.clip(q ** 3.0, 0, None)
            sig, kap = 3.0 * f, np.ones(len(l))
            b = np.exp(-dt * sig / kap)
            c = np.where(b == 1, 0.0, (b - 1) * sig / np.where(sig > 0, sig * kap, 1.0))
            sl = slice(0, wd) if side == 0 else slice(N - wd + l[0], N)
            if side == 0:
                b, c = b[::-1], c[::-1]
            shape = [1, 1, 1]
            shape[dim] = len(l)
            idx = [slice(None)] * 3
            idx[dim] = sl
            self.parts.append([tuple(idx)] + [torch.tensor(np.ascontiguousarray(v), device=_dev())
                                              .reshape(shape) for v in (b, c)] + [{}])

    def __call__(self, name, D):
        for idx, b, c, psi in self.parts:
            v = D[idx]
            psi[name] = c * v + (b * psi[name] if name in psi else 0.0)
            v += psi[name]
        return D


def _amp_phase(t, f):
    """Amplitude (>= 0) and phase of A sin(t + phase) + B from three samples."""
    s, c = [math.sin(v) for v in t], [math.cos(v) for v in t]
    f10, f21 = f[1] - f[0], f[2] - f[1]
    ph = torch.atan2(f10 * (s[2] - s[1]) - f21 * (s[1] - s[0]),
                     f21 * (c[1] - c[0]) - f10 * (c[2] - c[1]))
    hi = f21 / (torch.cos(ph) * (s[2] - s[1]) + torch.sin(ph) * (c[2] - c[1]))
    lo = f10 / (torch.cos(ph) * (s[1] - s[0]) + torch.sin(ph) * (c[1] - c[0]))
    A = torch.where(f21 * f21 >= f10 * f10, hi, lo)
    zero = (f10 == 0) & (f21 == 0)
    A, ph = torch.where(zero, 0.0, A), torch.where(zero, 0.0, ph)
    neg = A < 0
    return torch.where(neg, -A, A), torch.where(neg, ph + math.pi, ph)


def _torch_solve(case, p, adjoint=False):
    """The six phasors [Nz, Ny, Nx] (complex128 tensors) of a solve of `case`."""
    Nx, Ny, Nz, d, wl = (case[k] for k in ("Nx", "Ny", "Nz", "d", "wl"))
    dev = _dev()
    R = wl / (2 * math.pi)
    dt = 0.95 * d / R / math.sqrt(3)
    r = R / d
    tn = int(wl / d * math.sqrt(3) * 3 / 4)
    w = _pml(case)
    sizes = (Nx, Ny, Nz)
    ax = {f: [_Axis(a, sizes[a], w[2 * a:2 * a + 2], dt, f == "H", 2 - a) for a in range(3)]
          for f in "HE"}
    lossy = case["loss"] > 0
    a, b, m = [], [], []
    for e in p["mats"][:3]:
        e = torch.tensor(e, device=dev, dtype=torch.complex128)
        if lossy:
            er, ei = e.real / dt, e.imag * 0.5
            a.append((er - ei) / (er + ei))
            b.append(1.0 / (er + ei))
        else:
            b.append(dt / e.real)
    mu_one = case["mu"] == 1.0
    for v in p["mats"][3:]:
        m.append(dt if mu_one else dt / torch.tensor(v.real.copy(), device=dev))
    src, (k1, k2, j1, j2, i1, i2) = p["adj" if adjoint else "fwd"]
    box = (slice(i1, i2), slice(j1, j2), slice(k1, k2))
    src = [torch.tensor(v, device=dev) for v in src]
    T, mn = RAMP, 1e-4
    kk = T * T / math.log((1 + mn) / mn)

    def current(c, t):
        env = (1 + mn) * math.exp(-(t - T) ** 2 / kk) - mn if t <= T else 1.0
        return env * (math.sin(t) * src[c].real - math.cos(t) * src[c].imag)

    E = [torch.zeros((Nz, Ny, Nx), device=dev, dtype=torch.float64) for _ in range(3)]
    H = [torch.zeros_like(E[0]) for _ in range(3)]
    sign = [{"0": 0.0, "E": -1.0, "H": 1.0}[v] for v in case["bc"]]

    def fwd(F, axis):                       # forward difference, zero past the max face
        dim = 2 - axis
        o = torch.empty_like(F)
        n = F.shape[dim]
        torch.sub(F.narrow(dim, 1, n - 1), F.narrow(dim, 0, n - 1), out=o.narrow(dim, 0, n - 1))
        torch.neg(F.narrow(dim, n - 1, 1), out=o.narrow(dim, n - 1, 1))
        return o.mul_(r)

    def bwd(F, axis):                       # backward difference, mirror at the min face
        dim = 2 - axis
        o = torch.empty_like(F)
        n = F.shape[dim]
        torch.sub(F.narrow(dim, 1, n - 1), F.narrow(dim, 0, n - 1), out=o.narrow(dim, 1, n - 1))
        torch.mul(F.narrow(dim, 0, 1), 1.0 - sign[axis], out=o.narrow(dim, 0, 1))
        return o.mul_(r)

    # (component, its two derivative terms (axis, field, sign))
    curl = ((0, (2, 1, 1.0), (1, 2, -1.0)), (1, (0, 2, 1.0), (2, 0, -1.0)),
            (2, (1, 0, 1.0), (0, 1, -1.0)))

    def step(n):
        t = n * dt
        for c, p1, p2 in curl:
            D = ax["H"][p1[0]]((c, 0), fwd(E[p1[1]], p1[0]))
            D.sub_(ax["H"][p2[0]]((c, 1), fwd(E[p2[1]], p2[0])))
            H[c].addcmul_(D, m[c]) if torch.is_tensor(m[c]) else H[c].add_(D, alpha=m[c])
        for c in range(3):
            mu = m[c][box] if torch.is_tensor(m[c]) else m[c]
            H[c][box] += current(3 + c, t) * mu
        t += 0.5 * dt
        for c, p1, p2 in curl:
            D = ax["E"][p2[0]]((c, 0), bwd(H[p2[1]], p2[0]))
            D.sub_(ax["E"][p1[0]]((c, 1), bwd(H[p1[1]], p1[0])))
            if lossy:
                E[c].mul_(a[c])
            E[c].addcmul_(D, b[c])
        for c in range(3):
            E[c][box] -= current(c, t) * b[c][box]

    n = 0
    if case["steps"]:
        for n in range(case["steps"]):
            step(n)
        n0 = case["steps"]
    else:
        # sample points of the padded grid; a face ghost reads the opposite face
        total = Nx * Ny * Nz
        cells = []
        for q in range(0, total, total // case["nconv"]):
            at = (q // ((Nx + 2) * (Ny + 2)), q // (Nx + 2) % (Ny + 2), q % (Nx + 2))
            N = (Nz, Ny, Nx)
            ghosts = sum(v == 0 or v == N[u] + 1 for u, v in enumerate(at))
            g = [(v - 1) % N[u] for u, v in enumerate(at)]
            cells.append(-1 if ghosts > 1 else (g[0] * Ny + g[1]) * Nx + g[2])
        cells = torch.tensor(cells, device=dev)
        live = (cells >= 0).double()
        cells = cells.clamp(min=0)
        f = [torch.zeros((3, len(cells)), device=dev, dtype=torch.float64) for _ in range(3)]
        ts = [0.0, 0.0, 0.0]
        A0 = P0 = torch.zeros(len(cells), device=dev, dtype=torch.float64)
        limit = wl / d * 500
        while True:
            step(n)
            if n % tn == tn - 1:
                f = f[1:] + [torch.stack([F.reshape(-1)[cells] * live for F in E])]
                ts = ts[1:] + [n * dt]
                A, P = _amp_phase(ts, f)
                A, P = A.sum(0), P.sum(0)
                ca, cp = (A - A0).norm() / A0.norm(), (P - P0).norm() / P0.norm()
                A0, P0 = A, P
                if ca <= RTOL and cp <= math.sqrt(RTOL):
                    break
            n += 1
            if n > limit:
                n -= 1
                break
        n0 = n + 1
    snaps = [[F.clone() for F in E + H]]
    for half in range(2):
        for q in range(n0 + half * tn, n0 + (half + 1) * tn):
            step(q)
        snaps.append([F.clone() for F in E + H])
    out = []
    for c in range(6):
        t = [(n0 + q * tn) * dt - (0.5 * dt if c > 2 else 0.0) for q in range(3)]
        A, P = _amp_phase(t, [s[c] for s in snaps])
        out.append(torch.complex(A * torch.cos(P), -A * torch.sin(P)))
    return out


# cells averaged onto the Ez position, per component, as (dz, dy, dx)
MEAN = (((0, 0, 0), (0, 0, -1), (1, 0, 0), (1, 0, -1)),
        ((0, 0, 0), (0, -1, 0), (1, 0, 0), (1, -1, 0)),
        ((0, 0, 0),), ((0, 0, 0), (0, -1, 0)), ((0, 0, 0), (0, 0, -1)),
        tuple((a, b, c) for a in (0, 1) for b in (0, -1) for c in (0, -1)))


def _interp(F, c, box):
    k1, k2, j1, j2, i1, i2 = box
    v = sum(F[c][i1 + a:i2 + a, j1 + b:j2 + b, k1 + e:k2 + e] for a, b, e in MEAN[c])
    return v / len(MEAN[c])


def _power(case, F):
    """Flux through the box one cell inside the CPML."""
    w, d = case["pml"], case["d"]
    N = (case["Nx"], case["Ny"], case["Nz"])
    lo = [int((w * d + d) / d) for _ in N]
    hi = [int(((n - 1) * d - w * d - d) / d) for n in N]
    P = 0.0
    terms = ((1, 5, 2, 4), (0, 5, 2, 3), (0, 4, 1, 3))
    for axis in range(3):
        flip = -1.0 if axis == 1 else 1.0
        for at, s in ((lo[axis], -1.0), (hi[axis], 1.0)):
            box = []
            for u in range(3):
                box += [at, at + 1] if u == axis else [lo[u], hi[u] + 1]
            a, b, c, e = (_interp(F, q, box) for q in terms[axis])
            P += flip * s * 0.5 * d * d * float((a * b.conj() - c * e.conj()).real.sum())
    return P


def exact(case, seed):
    kind = case["kind"]
    if kind in ("build", "gradient"):
        return None                       # polygon overlaps and the whole design loop
    if kind == "batch":
        out = []
        for c, m, adj in _members(case, seed):
            out += [f.cpu().numpy() for f in _torch_solve(c, _problem(c, m), adj)[:3]]
        return out
    p = _problem(case, seed)
    F = _torch_solve(case, p)
    if kind == "solve":
        n = case["Nx"] * case["Ny"] * case["Nz"]
        return [f.cpu().numpy() for f in (F if n < 2000000 else F[:3])]
    if kind == "fields":
        out = []
        for q in _planes(case):
            box = (q.k1, q.k2, q.j1, q.j2, q.i1, q.i2)
            out += [_interp(F, c, box).cpu().numpy() for c in range(6)]
        return out + [_power(case, F)]
    G = _torch_solve(case, p, adjoint=True)
    rng = np.random.default_rng([3, seed])
    pidx, comp, cell, deps = _entries(case, rng)
    A0, (k1, k2, j1, j2, i1, i2) = _ydax(case, p, rng)
    prod = torch.stack([(F[c] * G[c]).reshape(-1) for c in range(3)]).cpu().numpy()
    g = np.zeros(case["members"])
    np.add.at(g, pidx, -2 * np.real(1j * prod[comp, cell] * deps))
    y = 0.0
    for c in range(3):
        box = (slice(i1, i2), slice(j1, j2), slice(k1, k2))
        y += np.sum(1j * (p["mats"][c] - A0[c])[box] * prod[c].reshape(A0[c].shape)[box])
    return {"gradient": g, "ydAx": np.array([y])}
