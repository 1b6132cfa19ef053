"""Materials built where the solver reads them: a structured eps sampled on
the GPU into the solver's arrays (emf_build_structured) against the arrays the
host sampler gives, and the index of distinct eps triples, which is exact: the
fields with it are bit for bit those without it, at the sizes where its width
changes (65535 and 65536 triples) and where it stays off (2^20 and one more)."""
import warnings

import numpy as np
import pytest

from emopt_amd.fdtd import FDTD
from emopt_amd.grid import ConstantMaterial3D, Rectangle, StructuredMaterial3D
from tests.cases import random_case, span
from tests.test_gpu_material import SHIFTS, _random_structure
from tests.test_gpu_parity import _run_steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,m", [((61, 43, 29), 1), ((61, 43, 29), 2), ((61, 43, 29), 65535),
                                    ((61, 43, 29), 65536), ((61, 43, 29), 61 * 43 * 29),
                                    ((103, 101, 102), 1 << 20), ((103, 101, 102), (1 << 20) + 1)])
def test_index_is_exact(dims, m):
    case = random_case(*dims, w=(5, 4, 3, 6, 4, 5), seed=7, nsrc=2, mu_rand=False)
    n = dims[0] * dims[1] * dims[2]
    which = np.minimum(np.arange(n), m - 1)
    np.random.default_rng(m).shuffle(which)
    for c in range(3):
        step = (1, 3, 7)[c]
        case["mats"][c] = (2 + 1e-6 * (which // step)).astype(complex).reshape(dims[::-1])
    a = _run_steps(case, 7, kind=1, compress=1)
    b = _run_steps(case, 7, kind=1, compress=0)
    assert any(np.any(x != 0) for x in a)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


def _sim(N, d):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        return FDTD(span(N[0], d), span(N[1], d), span(N[2], d), d, d, d, 1.55)


@pytest.mark.parametrize("overlap", ["exact", "supersample"])
@pytest.mark.parametrize("N", [(40, 34, 26), (37, 33, 2), (2, 3, 25), (65, 31, 23)])
def test_build_in_place_equals_the_host_sampler(N, overlap):
    d = 0.05
    sim = _sim(N, d)
    for seed in (1, 2):
        eps, _ = _random_structure(seed, overlap=overlap)
        sim.set_materials(eps, ConstantMaterial3D(1.5 + 0.25j))
        assert sim._samples_in_place()
        sim.build()
        diag = sim.get_A_diag()
        for c, (sx, sy, sz) in enumerate(SHIFTS[:3]):
            host = eps.get_values(0, N[0], 0, N[1], 0, N[2], sx=sx, sy=sy, sz=sz).ravel()
            assert np.array_equal(diag[c], host), (seed, c)
        for c in range(3, 6):
            assert np.all(diag[c] == 1.5)


def test_a_refused_structure_leaves_the_materials():
    N, d = (20, 20, 6), 0.1
    sim = _sim(N, d)
    good, _ = _random_structure(1, overlap="exact")
    sim.set_materials(good, ConstantMaterial3D(1.0))
    sim.build()
    before = [a.copy() for a in sim.get_A_diag()]
    bad = StructuredMaterial3D(2.0, 2.0, 1.0, 0.1, 0.1, 0.1)
    for q in range(10):              # partial rectangles in one cell
        bad.add_primitive(Rectangle(1.0, 1.0, 1.0 - 0.01 * q, 1.0 + 0.013 * q, material_value=2.0,
                                    layer=q), 0.0, 1.0)
    sim.set_materials(bad, ConstantMaterial3D(1.0))
    with pytest.raises(Exception, match="more than 8 primitives"):
        sim.build()
    for a, b in zip(sim.get_A_diag(), before):
        assert np.array_equal(a, b)
