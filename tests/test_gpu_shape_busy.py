"""Shape derivatives of a solver that is a member of a batch: the host's."""
import numpy as np
import pytest

from emopt_amd import _lib
from emopt_amd.batch import Batch
from emopt_amd.grid import ConstantMaterial3D, Rectangle, StructuredMaterial3D
from emopt_amd.shape import boundary_deps, rect_edge_velocity
from tests.test_gpu_shape import D, N, _same, _sims

pytestmark = pytest.mark.gpu


def test_batch_member():
    eps = StructuredMaterial3D(*(n * D for n in N), D, D, D)
    p = Rectangle(0.5, 0.4, 0.43, 0.31, material_value=9.0, layer=1)
    eps.add_primitive(p, 0.0, 0.3)
    dev, host = _sims()
    dev.w_pml = [2.5 * D] * 6
    dev.set_materials(eps, ConstantMaterial3D(1.0))
    b = Batch()
    mid = b.add(dev, postprocess=False)
    with pytest.raises(_lib.EmfError) as err:
        dev._lib.emf_reset_pml(dev._h)
    assert err.value.code == _lib.ERR_STATE
    for x, y in zip(boundary_deps(dev, eps, p, rect_edge_velocity("xr")),
                    boundary_deps(host, eps, p, rect_edge_velocity("xr"))):
        assert len(x) > 0 and np.array_equal(x, y)
    b.remove(mid)
    b.close()
    assert _same(eps, p, rect_edge_velocity("xr")) > 0
