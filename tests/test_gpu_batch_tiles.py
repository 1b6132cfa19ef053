"""Batches whose members the graphs step, also those that would fit on chip (which
emf_set_resident turns off here): graphs, lanes, groups and the members' solve
loops against single solves with the step kernels, and batches of both kinds."""
import warnings

import pytest

import numpy as np

from tests.cases import all_fields, batch_case, build_sim, rel_l2
from tests.test_gpu_batch import SMALL, TOL
from tests.test_gpu_resident import _boxes

pytestmark = pytest.mark.gpu

KEYS = ("n0", "Tn", "steps", "status", "nchecks")


def _sim(case, resident=0, **limits):
    sim = build_sim(case)
    for key, value in limits.items():
        setattr(sim, key, value)
    sim._lib.emf_set_resident(sim._h, resident, 0)
    assert (_boxes(sim) > 0) == bool(resident)
    return sim


def _result(sim, case):
    return ({k: sim.last_solve[k] for k in KEYS}, np.array(sim.convergence_history),
            all_fields(sim, case, case["adjoint"]))


def _plain(case, **kw):
    sim = _sim(case, **kw)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        if case["adjoint"]:
            sim.solve_adjoint()
        else:
            sim._register(sim._sources)
            sim._solve(0)
    return _result(sim, case)


def _batch(cases, kws, until=(), **opts):
    from emopt_amd.batch import Batch
    b = Batch(**opts)
    sims = [_sim(c, **k) for c, k in zip(cases, kws)]
    for s, c in zip(sims, cases):
        b.add(s, adjoint=c["adjoint"], postprocess=False)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        for n in until:
            b.run(until="graphs", max_graphs=n)
        b.run()
    assert b.running == 0
    b.close()
    return [_result(s, c) for s, c in zip(sims, cases)]


def _agree(got, ref):
    assert got[0] == ref[0]
    np.testing.assert_allclose(got[1], ref[1], rtol=1e-8)
    errs = [rel_l2(x, y) for x, y in zip(got[2], ref[2])]
    assert max(errs) <= TOL, errs


def _same(got, ref):
    assert got[0] == ref[0] and np.array_equal(got[1], ref[1])
    assert all(np.array_equal(x, y) for x, y in zip(got[2], ref[2]))


@pytest.fixture(scope="module")
def cases():
    out = [batch_case(q, n_fwd=3, **SMALL) for q in range(5)]
    out[1]["nconv"] = 200                     # more sample points than lanes
    for q, bc in ((2, "0H0"), (3, "EEH")):    # symmetry faces, slabs of other widths
        out[q]["bc"] = bc
        out[q]["w"] = [0 if bc[a // 2] in "EH" and a % 2 == 0 else max(w - (a == 1), 2)
                       for a, w in enumerate(out[q]["w"])]
    return out


@pytest.fixture(scope="module")
def refs(cases):
    return [_plain(c) for c in cases]


@pytest.fixture(scope="module")
def alone(cases):
    return [_batch([c], [{}], steps_per_graph=16)[0] for c in cases]


def test_members_alone_match_single_solves(alone, refs):
    for got, ref in zip(alone, refs):
        _agree(got, ref)


@pytest.mark.parametrize("opts", [
    dict(steps_per_graph=16), dict(steps_per_graph=16, use_graph=False),
    dict(steps_per_graph=7, lanes=1, group=1), dict(steps_per_graph=32, lanes=3, group=1, rotate_groups=True),
    dict(steps_per_graph=16, lanes=2, group=2, rotate_groups=True), dict(steps_per_graph=16, group_bytes=0),
])
def test_together_as_alone(cases, alone, opts):
    """Graphs and direct launches, lanes and groups: the same to the bit."""
    opts = dict(opts)
    if "group" in opts:
        opts["group_bytes"] = opts.pop("group") * max(80 * c["Nx"] * c["Ny"] * c["Nz"] for c in cases)
    for until in ((), (11, 40)):
        for got, ref in zip(_batch(cases, [{}] * len(cases), until, **opts), alone):
            _same(got, ref)


@pytest.mark.parametrize("limits", [dict(fixed_n0=300), dict(fixed_n0=0), dict(Nmax=170.5), dict(Nmax=3)])
def test_limits(cases, limits):
    pair = [cases[0], cases[3]]
    for got, c in zip(_batch(pair, [limits] * 2, steps_per_graph=16), pair):
        _agree(got, _plain(c, **limits))


@pytest.mark.parametrize("until", [(), (5,), (60, 60)])
def test_both_kinds_in_one_batch(cases, alone, until):
    """Every other member on chip: each as alone, to the bit."""
    kws = [dict(resident=q % 2) for q in range(len(cases))]
    got = _batch(cases, kws, until, steps_per_graph=16)
    for q, c in enumerate(cases):
        _same(got[q], _plain(c, resident=1) if q % 2 else alone[q])
