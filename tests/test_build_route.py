"""Which materials the GPU samples in place: none whose samplers are replaced, by
a subclass or on the object itself (CPU only)."""
import numpy as np
import pytest

from emopt_amd.fdtd import FDTD
from emopt_amd.grid import ConstantMaterial3D, StructuredMaterial3D


def _sim(cls=FDTD):
    sim = object.__new__(cls)
    sim._h = None
    sim._eps = StructuredMaterial3D(1.0, 1.0, 1.0, 0.1, 0.1, 0.1)
    sim._mu = ConstantMaterial3D(1.0)
    return sim


def _values(*args, **kw):
    return np.ones(1000, dtype=complex)


def test_stock_samplers_are_sampled_in_place():
    assert _sim()._samples_in_place()


@pytest.mark.parametrize("owner,name", [
    ("sim", "_sample"), ("sim", "set_material_arrays"), ("_eps", "get_values"),
    ("_eps", "get_values_device"), ("_mu", "get_values")])
def test_samplers_replaced_on_the_object_are_asked(owner, name):
    sim = _sim()
    setattr(sim if owner == "sim" else getattr(sim, owner), name, _values)
    assert not sim._samples_in_place()


@pytest.mark.parametrize("name", ["_sample", "set_material_arrays"])
def test_samplers_replaced_by_a_subclass_are_asked(name):
    assert not _sim(type("Own", (FDTD,), {name: _values}))._samples_in_place()
