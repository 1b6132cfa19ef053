"""Results through pinned host memory: the sizes where the route changes (one
piece, several lanes with remainders, past a slab) give the same values."""
import numpy as np
import pytest

from tests.cases import build_sim, random_case

pytestmark = pytest.mark.gpu


def _solved(dims):
    case = random_case(*dims, w=(2,) * 6, seed=8, mu_rand=False)
    sim = build_sim(case)
    for s in sim._sources:
        sim._adj_sources.append(s)
    sim.fixed_n0 = 12
    sim._register(sim._sources)
    sim._solve(0)
    sim._solve(1)
    return sim, case


# complex values of a field: 1 MB is one piece, 8 MB a slab
@pytest.mark.parametrize("dims", [(64, 32, 32), (64, 32, 33), (101, 53, 37), (128, 64, 66),
                                  (131, 73, 67)])
def test_whole_fields_equal_their_planes(dims):
    from emopt_amd.misc import DomainCoordinates as D
    sim, case = _solved(dims)
    Nx, Ny, Nz = dims
    d = case["d"]
    whole = D.from_indices(0, Nx, 0, Ny, 0, Nz, d, d, d)
    for c in ("Ex", "Hz"):
        ref = np.concatenate([sim.get_field(c, D.from_indices(0, Nx, 0, Ny, i, i + 1, d, d, d))
                              for i in range(Nz)])
        assert np.any(ref != 0)
        assert np.array_equal(sim.get_field(c, whole), ref)
        part = D.from_indices(1, Nx, 0, Ny - 1, 0, Nz, d, d, d)
        assert np.array_equal(sim.get_field(c, part), ref[:, :Ny - 1, 1:])
    ex, hz = sim.get_field("Ex", whole), sim.get_field("Hz", whole)
    prod = sim.field_products(whole, "E")[0]
    ref = ex * sim.get_adjoint_field("Ex", whole)
    assert np.abs(prod - ref).max() <= 1e-15 * np.abs(ref).max()
    eps = sim.get_A_diag()
    for a, m in zip(eps, case["mats"]):
        assert np.array_equal(a, np.asarray(m).ravel())
    assert hz.shape == (Nz, Ny, Nx)


@pytest.mark.parametrize("n", [0, 1, 1000, 65537, 290000, 310000])
def test_gradient_entries_below_and_past_a_slab(n):
    """Segments with no entries, ungrouped input, one thread's and several
    threads' worth of entries, and more than a slab holds."""
    sim, case = _solved((40, 30, 20))
    rng = np.random.default_rng(n)
    N = 40 * 30 * 20
    npar = 7
    pidx = rng.choice([0, 1, 3, 4, 6], n).astype(np.int32)
    comp = rng.integers(0, 3, n).astype(np.int32)
    cell = rng.integers(0, N, n)
    deps = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    g = sim.grad_assemble(pidx, comp, cell, deps, npar, step=2.0)
    F = np.stack([np.ravel(_full(sim, c, case)) for c in ("Ex", "Ey", "Ez")])
    G = np.stack([np.ravel(_full(sim, c, case, True)) for c in ("Ex", "Ey", "Ez")])
    t = np.real(G[comp, cell] * 1j * deps * F[comp, cell])
    ref, mag = np.zeros(npar), np.zeros(npar)
    np.add.at(ref, pidx, -t)
    np.add.at(mag, pidx, np.abs(t))
    # sums of n terms in another order: n eps of the terms' magnitude bounds the difference
    assert np.all(np.abs(g - ref) <= max(n, 16) * 2.3e-16 * mag)
    assert g[2] == 0 and g[5] == 0


def _full(sim, c, case, adjoint=False):
    from emopt_amd.misc import DomainCoordinates as D
    dom = D.from_indices(0, case["Nx"], 0, case["Ny"], 0, case["Nz"], *([case["d"]] * 3))
    return sim.get_adjoint_field(c, dom) if adjoint else sim.get_field(c, dom)


def test_ydax_below_and_past_a_slab():
    sim, case = _solved((80, 70, 60))
    rng = np.random.default_rng(1)
    shp = (60, 70, 80)
    A0 = [np.asarray(m) + 1e-2 * rng.standard_normal(shp) for m in case["mats"][:3]]
    t = sum(_full(sim, c, case, True) * 1j * (np.asarray(m) - a) * _full(sim, c, case)
            for c, m, a in zip(("Ex", "Ey", "Ez"), case["mats"], A0))
    for box in ((0, 80, 0, 70, 0, 60), (3, 70, 5, 60, 7, 20), (4, 5, 6, 7, 8, 9)):
        k1, k2, j1, j2, i1, i2 = box
        v = t[i1:i2, j1:j2, k1:k2]
        got = sim.calc_ydAx(A0, box=box)
        assert abs(got - v.sum()) <= v.size * 2.3e-16 * np.abs(v).sum() + 1e-300
