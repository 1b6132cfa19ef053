"""Two-pass tiles in strips per XCD (a step's data within the Infinity Cache):
every cell exactly once, so fields bit for bit those of the plain tile order,
at grids with fewer tiles than XCDs, ragged strips (the last one shorter) and
every work-group shape, for all coefficient layouts."""
import numpy as np
import pytest

from tests.cases import random_case
from tests.test_gpu_parity import _run_steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 3, 2), (7, 5, 3), (64, 4, 1), (65, 49, 17), (70, 97, 11),
                                  (130, 100, 9)])
@pytest.mark.parametrize("kw", [{}, {"ceps": True}, {"mu_rand": True}])
def test_strips_cover_every_cell_once(dims, kw):
    w = tuple(min(3, (n - 1) // 2) for n in dims for _ in range(2))
    case = random_case(*dims, w=w, seed=5, nsrc=1, **{"mu_rand": False, **kw})
    ref = _run_steps(case, 9, kind=1, tyg=4, zc=2, order=0)
    for tyg, zc in ((4, 1), (4, 2), (1, 1), (2, 3), (8, 2)):
        got = _run_steps(case, 9, kind=1, tyg=tyg, zc=zc, order=3)
        for a, b in zip(got, ref):
            assert np.array_equal(a, b), (tyg, zc)
    for kind in (3, 4):
        got = _run_steps(case, 9, kind=kind, tyg=2, zc=1, order=3)
        for a, b in zip(got, ref):
            np.testing.assert_allclose(a, b, rtol=0, atol=1e-13 * max(np.abs(r).max() for r in ref))
